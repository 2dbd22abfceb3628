// m25x_tslu.hip - the tournament of a tournament-pivoting LU panel (k_tslu), built once per element type
// (M25X_TSLU_C64 set: complex64, else complex128) so the two unrolled instantiations compile in parallel.
#include <cstddef>
#include "m25x_lu_dev.h"

namespace m25x {
namespace lu {
namespace {

// GEPP of up to 256 rows of 64 columns by one workgroup, eight columns (a sub-panel) at a time. Eight row waves hold the
// rows in registers (two threads a row, lanes L and L + 32 of a wave; the thread of half h = lane / 32 has columns
// 2 j + h); four panel waves factor each sub-panel, a row a lane, the sub-panel passing through LDS. What bounds a GEPP
// is the chain of its 64 steps (search the column, fetch the pivot row, update), not arithmetic: on this machine a
// dependent instruction takes 8 cycles, a DPP round 16, a vector compare used by the scalar unit 28, an LDS hand-off
// between waves with its barrier about 110, an LDS write of 16 B 14 cycles of the LDS whatever lanes take part. So a
// step handles few rows and columns a lane and hands over one key a wave and one row. The row waves meanwhile apply the
// last sub-panel to the columns beyond the next one, one pivot between a step's two barriers, at a lower issue priority;
// only the next eight columns' update stays on the chain. Measured (64 steps of 256 rows): 88 us with every step spread
// over the workgroup's 64 columns, 47 us so (complex64); 112 and 52 us (complex128). A step takes about 1200 cycles,
// the hand-over from one sub-panel to the next 3500.
// Every element takes the same fused multiply-subtracts in the same order as an unblocked right-looking GEPP.
typedef unsigned long long u64;
constexpr int SPW = 8;                    // columns a sub-panel
constexpr int NSP = TW / SPW;
constexpr int RWV = 8, PWV = 4;           // row waves, panel waves
constexpr int NTH = 64 * (RWV + PWV);     // threads of the workgroup

template <typename T> struct GeppLds {
    T lp[2][SPW][Tour<T>::RL];            // a sub-panel's columns, then its multipliers (two, alternating)
    T us[SPW][2][TH];                     // its pivot rows' later columns (half h, column 2 j + h), then U12
    T prow[SPW][SPW];                     // its pivot rows of L \ U within it
    T rcp[SPW];                           // the reciprocals of its pivots
    int4 key[2][PWV];                     // the panel waves' best: magnitude words, position (two steps, alternating)
    T spare[PWV][SPW + 16 / sizeof(T)];   // where the rows that are not the best write: a key, or a row and its reciprocal
    int step_of[Tour<T>::RL];             // a pivot row's step, -1 before
};
// a key goes to the start of a spare row as one int4, whose place the compiler takes to be a multiple of 16 bytes
template <typename T> constexpr bool spare_aligned()
{
    return alignof(GeppLds<T>) >= sizeof(int4) && offsetof(GeppLds<T>, spare) % sizeof(int4) == 0 &&
           sizeof(GeppLds<T>::spare[0]) % sizeof(int4) == 0;
}
static_assert(spare_aligned<float2>() && spare_aligned<double2>(), "a spare row starts at 16 bytes");

// LDS traffic done, then the barrier: stores to global memory stay in flight across it
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// the wave's largest value, in a scalar register: DPP rounds within rows of 16 lanes, then across the rows (row_bcast),
// each one instruction (the exchange is the operation's source modifier, the old value the operation's identity)
#define M25X_MAXDPP(ctrl) v = max(v, __builtin_amdgcn_update_dpp((int)0x80000000, v, ctrl, 0xF, 0xF, false))
__device__ inline int quad_max(int v)
{
    M25X_MAXDPP(0xB1);       // quad_perm [1, 0, 3, 2]
    M25X_MAXDPP(0x4E);       // quad_perm [2, 3, 0, 1]
    return v;
}
__device__ inline int wave_max(int v)
{
    v = quad_max(v);
    M25X_MAXDPP(0x141);      // row_half_mirror
    M25X_MAXDPP(0x140);      // row_mirror
    M25X_MAXDPP(0x142);      // row_bcast:15
    M25X_MAXDPP(0x143);      // row_bcast:31
    return __builtin_amdgcn_readlane(v, 63);
}
#undef M25X_MAXDPP

// the number of lanes where c holds
__device__ __forceinline__ int lanes_with(bool c)
{
    int n = __builtin_popcountll(__builtin_amdgcn_ballot_w64(c));
    asm("" : "+s"(n));
    return n;
}

// The search orders rows by magnitude |Re| + |Im| (a NaN as zero), which is never negative, so the IEEE bits order as
// integers: the leading word (complex64: the whole magnitude) and, for complex128, the second.
__device__ inline void mag_words(float re, float im, int &hi, unsigned &lo)
{
    hi = __float_as_int(__builtin_fmaxf(fabsf(re) + fabsf(im), 0.0f));
    lo = 0;
}
__device__ inline void mag_words(double re, double im, int &hi, unsigned &lo)
{
    const long long b = __double_as_longlong(__builtin_fmax(fabs(re) + fabs(im), 0.0));
    hi = (int)(b >> 32);
    lo = (unsigned)b;
}

// A panel wave's share of a sub-panel (steps kb .. kb + 7, while < npiv; FULL: all eight): its lane's row's eight
// columns in lp, which holds the rows' multipliers on return. w: the wave (0 .. 3); pos: the row's position in the
// elimination order (rows never move; ties go to the earliest position, LAPACK's rule); cap: the largest leading word it
// may show in the search (negative, and the lane's own, once it is a pivot or where there is no row).
// A step: each wave's best row by DPP, its key to LDS; a barrier; every wave finds the best of the four keys; the row that
// has it publishes its later columns and its pivot's reciprocal (each lane has formed its own, in the shadow of the DPP
// rounds); a barrier; every lane updates its row. Both barriers are the row waves' too. An LDS write of 16 B takes 14
// cycles whatever lanes are in it, so only the winner writes a row; the other lanes' writes go to a spare place, which
// costs less than a branch around them.
template <typename T, bool FULL>
__device__ __forceinline__ void panel_factor(T (*lp)[Tour<T>::RL], GeppLds<T> &sh, int *order, int w, int &pos, int &cap,
                                             int kb, int npiv)
{
    typedef typename CX<T>::R R;
    constexpr bool WORD = sizeof(T) == 16;
    const int lane = threadIdx.x & 63, row = 64 * w + lane;
    int mine_at = -1;
    R re[SPW], im[SPW];
#pragma unroll
    for (int c = 0; c < SPW; ++c) {
        const T v = lp[c][row];
        re[c] = v.x; im[c] = v.y;
    }
    auto step = [&](auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value;
        if (!FULL && kb + k >= npiv) return;
        int hi;
        unsigned lo;
        mag_words(re[k], im[k], hi, lo);
        hi = min(hi, cap);
        bool in = hi == wave_max(hi);
        // the reciprocal conj(pv) / |pv|^2, as LAPACK's getf2 scales by 1 / pivot (1 for a zero pivot: it leaves the
        // column as it is)
        const R d = re[k] * re[k] + im[k] * im[k];
        const bool nz = d != (R)0;
        const R inv = (R)1 / d;
        const T rc = CX<T>::make(nz ? re[k] * inv : (R)1, nz ? -im[k] * inv : (R)0);
        const int lw = (int)(lo ^ 0x80000000u);              // the second word, ordered as signed
        int4 *const slot = &sh.key[k & 1][w], *const aside = (int4 *)&sh.spare[w][0];
        const int4 mine = make_int4(hi, lw, -1 - pos, 0);
        *(in ? slot : aside) = mine;
        if (lanes_with(in) != 1) {      // (looked at while the write is under way) the largest second word, then the
            if constexpr (WORD) {       // earliest position
                const int v = in ? lw : (int)0x80000000, best = wave_max(v);
                in = in && v == best;
            }
            const int v = in ? -1 - pos : (int)0x80000000, best = wave_max(v);
            in = in && v == best;
            *(in ? slot : aside) = mine;
        }
        lds_barrier();
        const int4 q = sh.key[k & 1][lane & 3];
        bool kin = q.x == quad_max(q.x);
        if (lanes_with(kin) != 16) {
            if constexpr (WORD) {
                const int v = kin ? q.y : (int)0x80000000, best = quad_max(v);
                kin = kin && v == best;
            }
            const int v = kin ? q.z : (int)0x80000000, best = quad_max(v);
            kin = kin && v == best;
        }
        const int bw = __builtin_ctz((unsigned)__builtin_amdgcn_ballot_w64(kin));
        const bool win = in && bw == w;
        if (bw == w) {
            T *to = win ? &sh.prow[k][0] : &sh.spare[w][0];
#pragma unroll
            for (int c = 0; c < SPW; ++c) to[c] = CX<T>::make(re[c], im[c]);
            *(win ? &sh.rcp[k] : &sh.spare[w][SPW]) = rc;
        }
        cap = win ? -1 - lane : cap;    // it leaves the search
        mine_at = win ? k : mine_at;
        const int p = -1 - __builtin_amdgcn_readlane(q.z, bw);
        pos = pos == kb + k ? p : pos;
        lds_barrier();
        const T l = tmul(CX<T>::make(re[k], im[k]), sh.rcp[k]);
        re[k] = l.x; im[k] = l.y;       // rows that are pivots already take part, their values no longer used
#pragma unroll
        for (int c = k + 1; c < SPW; ++c) {
            const T v = tfms(CX<T>::make(re[c], im[c]), l, sh.prow[k][c]);
            re[c] = v.x; im[c] = v.y;
        }
    };
    Unroll<0, SPW>::run(step);
    if (mine_at >= 0) {
        sh.step_of[row] = kb + mine_at;
        order[kb + mine_at] = row;
    }
#pragma unroll
    for (int c = 0; c < SPW; ++c) lp[c][row] = CX<T>::make(re[c], im[c]);
}

// U12 of a sub-panel (kb its first column): its pivot rows' later columns in us less the multiples of the rows before
// them, four lanes a column (lane q of a quad has rows q and q + 4; a row's final value reaches the others by a
// quad_perm broadcast), 16 columns a panel wave. top: the root's block, or NULL. The multipliers are read before the
// barrier that us waits for, which this takes (B).
template <int Q> __device__ __forceinline__ float quad_bcast(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), Q * 0x55, 0xF, 0xF, true));
}
template <int Q> __device__ __forceinline__ double quad_bcast(double v)
{
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)b, Q * 0x55, 0xF, 0xF, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(b >> 32), Q * 0x55, 0xF, 0xF, true);
    return __longlong_as_double((long long)((u64)hi << 32 | lo));
}
template <typename T>
__device__ __forceinline__ void panel_u12(GeppLds<T> &sh, int w, int kb, int nc, T *top)
{
    const T zero = CX<T>::make(0, 0);
    const int lane = threadIdx.x & 63, q = lane & 3, c = kb + SPW + 16 * w + (lane >> 2);
    T la[3], lb[SPW - 1];
#pragma unroll
    for (int i = 0; i < 3; ++i) la[i] = csel(i < q, sh.prow[q][i], zero);
#pragma unroll
    for (int i = 0; i < SPW - 1; ++i) lb[i] = csel(i < q + 4, sh.prow[q + 4][i], zero);
    lds_barrier();                              // B: the pivot rows' later columns are in LDS
    if (c < TW) {
        T a = sh.us[q][c & 1][c >> 1], b = sh.us[q + 4][c & 1][c >> 1];
        auto up = [&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value;
            const T u = CX<T>::make(quad_bcast<i & 3>(i < 4 ? a.x : b.x), quad_bcast<i & 3>(i < 4 ? a.y : b.y));
            if constexpr (i < 3) a = tfms(a, la[i], u);
            b = tfms(b, lb[i], u);
        };
        Unroll<0, SPW - 1>::run(up);
        sh.us[q][c & 1][c >> 1] = a;
        sh.us[q + 4][c & 1][c >> 1] = b;
        if (top) {
            top[c * TW + kb + q] = csel(c < nc, a, zero);
            top[c * TW + kb + q + 4] = csel(c < nc, b, zero);
        }
    }
}

// x[J + q] -= l u[q] for q < 4: the four columns' pivot-row values are those of lanes N .. N + 3 of each 16-lane row
// (u: a lane's value is column 16 g + lane % 16 of its half), broadcast by the multiply-add itself (row_newbcast, the
// one DPP control that 64-bit operations take too). Written out because the compiler does not fold a 64-bit broadcast
// into the operation, and a broadcast through LDS reads costs as much LDS time as the multiply-adds take. The s_nop
// covers the two wait states between a vector write of u and its DPP read. The same products in the same order as
// tfms.
template <int N> __device__ __forceinline__ void fms4(float *xr, float *xi, float2 u, float2 l)
{
#define M25X_FMS(R, I, n)                                                                                     \
    "v_fmac_f32_dpp %" #R ", %9, %11 row_newbcast:%c" #n " row_mask:0xf bank_mask:0xf\n"                      \
    "v_fmac_f32_dpp %" #I ", %9, -%10 row_newbcast:%c" #n " row_mask:0xf bank_mask:0xf\n"                     \
    "v_fmac_f32_dpp %" #R ", %8, -%10 row_newbcast:%c" #n " row_mask:0xf bank_mask:0xf\n"                     \
    "v_fmac_f32_dpp %" #I ", %8, -%11 row_newbcast:%c" #n " row_mask:0xf bank_mask:0xf\n"
    asm("s_nop 1\n" M25X_FMS(0, 4, 12) M25X_FMS(1, 5, 13) M25X_FMS(2, 6, 14) M25X_FMS(3, 7, 15)
        : "+v"(xr[0]), "+v"(xr[1]), "+v"(xr[2]), "+v"(xr[3]), "+v"(xi[0]), "+v"(xi[1]), "+v"(xi[2]), "+v"(xi[3])
        : "v"(u.x), "v"(u.y), "v"(l.x), "v"(l.y), "n"(N), "n"(N + 1), "n"(N + 2), "n"(N + 3));
#undef M25X_FMS
}
template <int N> __device__ __forceinline__ void fms4(double *xr, double *xi, double2 u, double2 l)
{
#define M25X_FMS(R, I, n)                                                                                     \
    "v_fmac_f64_dpp %" #R ", %9, %11 row_newbcast:%c" #n " row_mask:0xf bank_mask:0xf\n"                      \
    "v_fmac_f64_dpp %" #I ", %9, -%10 row_newbcast:%c" #n " row_mask:0xf bank_mask:0xf\n"                     \
    "v_fmac_f64_dpp %" #R ", %8, -%10 row_newbcast:%c" #n " row_mask:0xf bank_mask:0xf\n"                     \
    "v_fmac_f64_dpp %" #I ", %8, -%11 row_newbcast:%c" #n " row_mask:0xf bank_mask:0xf\n"
    asm("s_nop 1\n" M25X_FMS(0, 4, 12) M25X_FMS(1, 5, 13) M25X_FMS(2, 6, 14) M25X_FMS(3, 7, 15)
        : "+v"(xr[0]), "+v"(xr[1]), "+v"(xr[2]), "+v"(xr[3]), "+v"(xi[0]), "+v"(xi[1]), "+v"(xi[2]), "+v"(xi[3])
        : "v"(u.x), "v"(u.y), "v"(l.x), "v"(l.y), "n"(N), "n"(N + 1), "n"(N + 2), "n"(N + 3));
#undef M25X_FMS
}

// The thread's columns J0 .. J1 - 1 (multiples of four) updated by pivot jp of a sub-panel: its multiplier l, the
// pivot row's values (U12) from LDS.
template <typename T, int J0, int J1>
__device__ __forceinline__ void row_update(RowH<T> &x, T l, const T *us, int l16)
{
    if constexpr (J0 < J1 && J0 < 16) {
        const T u = us[l16];
        auto upd = [&](auto qc) __attribute__((always_inline)) {
            constexpr int j = J0 + 4 * decltype(qc)::value;
            fms4<j>(x.re + j, x.im + j, u, l);
        };
        Unroll<0, ((J1 < 16 ? J1 : 16) - J0) / 4>::run(upd);
    }
    if constexpr (J0 < J1 && J1 > 16) {
        constexpr int B = J0 > 16 ? J0 : 16;
        const T u = us[16 + l16];
        auto upd = [&](auto qc) __attribute__((always_inline)) {
            constexpr int j = B + 4 * decltype(qc)::value;
            fms4<j - 16>(x.re + j, x.im + j, u, l);
        };
        Unroll<0, (J1 - B) / 4>::run(upd);
    }
}

// GEPP of nr rows over columns [0, nc), the row thread's row (where have) at src with its columns lda apart: order[k] =
// the k-th pivot row. top (the tree's root only, else NULL): the pivot rows' L \ U as a column-major TW x TW block,
// rows [0, min(nr, nc)). Returns min(nr, nc).
template <typename T>
__device__ __forceinline__ int reg_gepp(bool have, const T *src, long lda, int nr, int nc, int *order,
                                        GeppLds<T> &sh, T *top)
{
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int npiv = nr < nc ? nr : nc;
    const T zero = CX<T>::make(0, 0);
    if (wv >= RWV) {                            // the panel waves: their chain issues ahead of the row waves' updates
        __builtin_amdgcn_s_setprio(3);
        const int w = wv - RWV, row = 64 * w + lane;
        int pos = row, cap = row < nr ? 0x7fffffff : -1 - lane;
        sh.step_of[row] = -1;
        lds_barrier();                          // the first sub-panel's columns are in LDS
        for (int s = 0; s * SPW < npiv; ++s) {
            const int kb = s * SPW;
            if (kb + SPW <= npiv) panel_factor<T, true>(sh.lp[s & 1], sh, order, w, pos, cap, kb, npiv);
            else panel_factor<T, false>(sh.lp[s & 1], sh, order, w, pos, cap, kb, npiv);
            lds_barrier();                      // A: multipliers and pivot rows out, the last update done
            if (top && w == 1) {
                const int j = lane >> 3, c = lane & 7;
                if (kb + j < npiv) top[(kb + c) * TW + kb + j] = csel(kb + c < nc, sh.prow[j][c], zero);
            }
            if (kb + SPW >= npiv) break;
            panel_u12<T>(sh, w, kb, nc, top);   // (takes barrier B)
            lds_barrier();                      // C: U12 out
            lds_barrier();                      // D: the next sub-panel's columns are in LDS
        }
        lds_barrier();
        return npiv;
    }
    const int row = wv * 32 + (lane & 31), h = lane >> 5;
    RowH<T> x;
    {
        long st = 2 * lda;
        asm volatile("" : "+s"(st));            // 32 addresses stepped, not kept in registers across the tree's levels
        const T *p = src + h * lda;
        auto ld = [&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            x.set(j, ldz(have && 2 * j + h < nc, p));
            p += st;
        };
        Unroll<0, TH>::run(ld);
    }
#pragma unroll
    for (int i = 0; i < SPW / 2; ++i) sh.lp[0][2 * i + h][row] = x.get(i);
    lds_barrier();
    bool more = true;
    auto sub = [&](auto sc) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value, kb = s * SPW, J = (s + 1) * (SPW / 2), JN = J + SPW / 2;
        if (!more) return;
        // the thread's places in LDS computed anew for each sub-panel: kept for all of them they go to scratch memory
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int row = (tid >> 6) * 32 + (tid & 31), h = (tid >> 5) & 1, l16 = tid & 15;
        const int nst = npiv - kb < SPW ? npiv - kb : SPW;
#pragma unroll 1
        for (int jp = 0; jp < nst; ++jp) {      // the panel waves' steps; meanwhile the last sub-panel's pivots
            lds_barrier();
            if constexpr (s > 0 && J < TH) row_update<T, J, TH>(x, sh.lp[(s & 1) ^ 1][jp][row], sh.us[jp][h], l16);
            lds_barrier();
        }
        if constexpr (s > 0 && J < TH)
            for (int jp = nst; jp < SPW; ++jp) row_update<T, J, TH>(x, sh.lp[(s & 1) ^ 1][jp][row], sh.us[jp][h], l16);
        lds_barrier();                          // A
        if (top) {                              // the rows that become pivots later keep their multipliers
#pragma unroll
            for (int i = 0; i < SPW / 2; ++i) x.set(s * (SPW / 2) + i, sh.lp[s & 1][2 * i + h][row]);
        }
        if (kb + SPW >= npiv) { more = false; return; }
        if constexpr (J < TH) {
            const int st = sh.step_of[row] - kb;
            if (st >= 0) {                      // a pivot of this sub-panel: its later columns out
                auto pub = [&](auto jc) __attribute__((always_inline)) {
                    constexpr int j = decltype(jc)::value;
                    sh.us[st][h][j] = x.get(j);
                };
                Unroll<J, TH>::run(pub);
            }
            lds_barrier();                      // B
            lds_barrier();                      // C
#pragma unroll
            for (int jp = 0; jp < SPW; ++jp) row_update<T, J, JN>(x, sh.lp[s & 1][jp][row], sh.us[jp][h], l16);
#pragma unroll
            for (int i = 0; i < SPW / 2; ++i) sh.lp[(s & 1) ^ 1][2 * i + h][row] = x.get(J + i);
            lds_barrier();                      // D
        }
    };
    Unroll<0, NSP>::run(sub);
    if (top) {                                  // a pivot row's multipliers of the sub-panels before its own
        const int st = sh.step_of[row];
        const int before = st >= 0 ? (st / SPW) * (SPW / 2) : 0;
        auto put = [&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value;
            if (j < before) top[(2 * j + h) * TW + st] = x.get(j);
        };
        Unroll<0, TH - SPW / 2>::run(put);
    }
    lds_barrier();
    return npiv;
}

// an int that another workgroup of the launch reads, or wrote
__device__ __forceinline__ void put_word(int *p, int v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int get_word(const int *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The tournament of panel [j0, j0 + jb) over rows [j0, n). Leaves: blockIdx.x (P of them) of RL rows. A node takes its
// children's nominees straight from A, which the launch leaves untouched: only their row numbers pass between
// workgroups. The root writes the panel's L11 \ U11 (top, column-major TW x TW), the interchanges (ipiv[j0 .. j0 + jb),
// LAPACK's convention) and the row moves they make as (destination, source) pairs (pairs[0] = count), and info for
// a zero pivot.
template <typename T>
__device__ __forceinline__ void tslu_body(const T *A, long lda, long n, long j0, int jb, int P, TNode<T> *nodes,
                                          int *arrive, T *top, int *ipiv, int *pairs, int *info, int leaf)
{
    constexpr int RL = Tour<T>::RL, AR = Tour<T>::AR;
    __shared__ GeppLds<T> gl;
    __shared__ int ids[RL];
    __shared__ int order[TW];
    __shared__ int go, counts[AR];
    const int t = threadIdx.x, lane = t & 63;
    const int row = (t >> 6) * 32 + (lane & 31), h = lane >> 5;     // row waves; from RL on in the panel waves
    int idx = leaf;
    const long r0 = j0 + (long)idx * RL;
    int nr = (int)std::min((long)RL, n - r0);
    bool have = row < nr;                       // the thread's row of the node: its entry of the panel's first column
    const T *src = A + j0 * lda + std::min(r0 + row, n - 1);
    if (t < nr) ids[t] = (int)(r0 + t);
    int lsize = P, loff = 0;
    for (;;) {
        const bool root = lsize == 1;           // only the root's factors are kept
        const int cnt = reg_gepp<T>(have, src, lda, nr, jb, order, gl, root ? top : (T *)nullptr);
        if (root) break;
        int parent = idx / AR, nchild = std::min(AR, lsize - parent * AR);
        while (nchild == 1) {                   // a node with one child nominates the child's rows unchanged
            loff += lsize;
            lsize = (lsize + AR - 1) / AR;
            idx = parent;
            parent = idx / AR;
            nchild = std::min(AR, lsize - parent * AR);
        }
        const int poff = loff + lsize, first = parent * AR;
        // Nominate: this node's pivot rows. They pass between workgroups as device-scope words, which go past the caches,
        // each wave waiting for its own before the workgroup counts itself in: a device-scope fence instead writes
        // back and drops a whole L2, which waits for whatever else is dirty there (beside a trailing update or a copy
        // a tournament took 1.5 to 1.8 times as long with three fences a level) and costs the update its tiles.
        TNode<T> *nd = nodes + loff + idx;
        if (t == 0) put_word(&nd->count, cnt);
        if (t < cnt) put_word(&nd->id[t], ids[order[t]]);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (t == 0) {
            const int old = __hip_atomic_fetch_add(arrive + poff + parent, 1, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
            go = old == nchild - 1;
            if (go) __hip_atomic_store(arrive + poff + parent, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (!go) return;
        // the last child to arrive factors the node: its children's nominees stacked in child order
        const TNode<T> *c0n = nodes + loff + first;
        if (t < nchild) counts[t] = get_word(&c0n[t].count);
        __syncthreads();
        int ch = 0, i = row;
        nr = 0;
        for (int q = 0; q < nchild; ++q) nr += counts[q];
        while (ch < nchild - 1 && i >= counts[ch]) { i -= counts[ch]; ++ch; }
        have = row < nr;
        const int id = have ? get_word(&c0n[ch].id[i]) : (int)r0;
        src = A + j0 * lda + id;
        if (have && h == 0) ids[row] = id;
        loff = poff;
        lsize = (lsize + AR - 1) / AR;
        idx = parent;
    }
    // the root: cnt == jb pivot rows, L11 \ U11 in top
    for (int e = t; e < TW * (TW - jb); e += NTH) {          // identity padding of a short last panel
        const int i = jb + e / TW, c = e % TW;
        top[c * TW + i] = CX<T>::make(i == c, 0);
    }
    __syncthreads();
    if (t == 0 && info) {
        for (int k = 0; k < jb; ++k) {
            const T d = top[k * TW + k];
            if (d.x == 0 && d.y == 0) {
                if (*info == 0) *info = (int)(j0 + k) + 1;
                break;
            }
        }
    }
    if (t < 64) {
        // LAPACK's interchanges: winner k to position j0 + k in order. Rows below the panel's first jb move only
        // when they win; lane i tracks loc (the position of the row first at j0 + i) and cont (the row at j0 + i).
        const int i = t;
        const int top_end = (int)j0 + jb;
        int loc = (int)j0 + i, cont = (int)j0 + i;
        const int win = i < jb ? ids[order[i]] : 0;
        for (int k = 0; k < jb; ++k) {
            const int w = __builtin_amdgcn_readlane(win, k);
            const int tpos = (int)j0 + k;
            const int pw = w < top_end ? __builtin_amdgcn_readlane(loc, w - (int)j0) : w;
            if (i == 0) ipiv[tpos] = pw;
            if (pw != tpos) {
                const int x = __builtin_amdgcn_readlane(cont, k);        // a row first in the panel's top
                if (i == k) cont = w;
                if (w < top_end && i == w - (int)j0) loc = tpos;
                if (pw < top_end && i == pw - (int)j0) cont = x;
                if (i == x - (int)j0) loc = pw;
            }
        }
        // the moves: position j0 + i takes row cont; a row of the top that ended below takes its place there
        const bool mv_top = i < jb && cont != (int)j0 + i;
        const bool mv_low = i < jb && loc >= top_end;
        const unsigned long long m1 = __ballot(mv_top), m2 = __ballot(mv_low);
        const unsigned long long below = (1ull << i) - 1;
        const int n1 = __popcll(m1);
        if (mv_top) {
            const int q = __popcll(m1 & below);
            pairs[1 + 2 * q] = (int)j0 + i;
            pairs[2 + 2 * q] = cont;
        }
        if (mv_low) {
            const int q = n1 + __popcll(m2 & below);
            pairs[1 + 2 * q] = loc;
            pairs[2 + 2 * q] = (int)j0 + i;
        }
        if (i == 0) pairs[0] = n1 + __popcll(m2);
    }
}

template <typename T>
__global__ __launch_bounds__(NTH) void k_tslu(const T *A, long lda, long n, long j0, int jb, int P,
                                                         TNode<T> *nodes, int *arrive, T *top, int *ipiv, int *pairs,
                                                         int *info)
{
    __builtin_amdgcn_s_setprio(2);    // ahead of the trailing update's waves where the LU's look-ahead runs it beside
    tslu_body<T>(A, lda, n, j0, jb, P, nodes, arrive, top, ipiv, pairs, info, blockIdx.x);
}

// item blockIdx.y of a batch; leaves past its own count, and items already factored, leave at once
template <typename T>
__global__ __launch_bounds__(NTH) void k_tslu_b(const m25x_lu_item *items, long j0)
{
    const m25x_lu_item it = items[blockIdx.y];
    const long n = it.n;
    if (j0 >= n) return;
    const int jb = (int)std::min((long)TW, n - j0);
    const int P = (int)tour_leaves(n - j0, Tour<T>::RL);
    if ((int)blockIdx.x >= P) return;
    const TourWork<T> w = tour_carve<T>(it.work, n);
    tslu_body<T>((const T *)it.A, it.lda, n, j0, jb, P, w.nodes, w.arrive, w.top, it.ipiv, w.pairs, it.info,
                 blockIdx.x);
}

}  // namespace

#ifdef M25X_TSLU_C64
typedef float2 TT;
#else
typedef double2 TT;
#endif

int launch_tslu(const TT *A, long lda, long n, long j0, int jb, int P, TNode<TT> *nodes, int *arrive, TT *top,
                int *ipiv, int *pairs, int *info, hipStream_t s)
{
    hipLaunchKernelGGL(k_tslu<TT>, dim3(P), dim3(NTH), 0, s, A, lda, n, j0, jb, P, nodes, arrive, top, ipiv,
                       pairs, info);
    return check_launch("getrf/tournament");
}

int launch_tslu_b(const TT *, const m25x_lu_item *items, int nitems, long j0, int Pmax, hipStream_t s)
{
    hipLaunchKernelGGL(k_tslu_b<TT>, dim3(Pmax, nitems), dim3(NTH), 0, s, items, j0);
    return check_launch("getrf_batched/tournament");
}

}  // namespace lu
}  // namespace m25x
