// m25x_lu.hip - dense complex LU on gfx950, and the triangular solves with its factor.
//
// A is column-major (the row-major Z of the reference seen as A = Z^T, the layout of scipy's lu_factor(Z.T)).
// Blocked right-looking. Two pivoting strategies:
// Partial pivoting (LAPACK's pivots exactly), panels of NB columns:
//   panel   one cooperative launch per panel: each workgroup keeps a slab of the panel's rows in LDS; every column
//           costs one grid barrier (pivot search, row interchange, scaling and the panel's rank-1 update in
//           between, the next column's candidates published before the barrier); pivots by LAPACK's rule
//           (largest |Re| + |Im|, the first on ties)
//   laswp   the panel's interchanges on the columns left and right of it
//   trsm    U12 = L11^-1 A12 (unit lower, forward substitution, one workgroup per 16 columns: k_trsm, these panels
//           only)
//   gemm    A22 -= A21 U12 on the matrix cores: complex products as real ones through the real embedding
//           (Re C = [Re A, Im A] [Re B; -Im B], Im C = [Re A, Im A] [Im B; Re B]), v_mfma_f64_16x16x4 for
//           complex128 and v_mfma_f32_16x16x4 for complex64 (FP32 accumulation)
// Tournament pivoting (CALU), panels of TW = 64 columns: the panel's pivots by a tree of GEPPs in one launch with no
// grid barrier (k_tslu), its row moves on every column (k_apply_moves), then L21 = A21 U11^-1 and U12 = L11^-1 A12 by
// substitution (k_tri) and A22 -= L21 U12 on the matrix cores (complex64 in FP32, or with FP64 accumulation where
// asked for); the next panel's tournament runs beside the larger updates.
// The solves (getrs): both triangles in one launch, one workgroup per 64-row diagonal block, triangle and two
// right-hand sides; each accumulates the products of its rows with the earlier blocks as their values appear, then
// solves its own block and hands its values on as self-marking words.
#include <atomic>
#include <mutex>
#include <vector>
#include "m25x_lu_dev.h"

using namespace m25x;
using namespace m25x::lu;

namespace {

template <typename T> constexpr int dtype_of() { return sizeof(T) == 16 ? M25X_C128 : M25X_C64; }

// ---- grid barrier (all workgroups of a cooperative launch co-resident) -------------------------------------
struct Bar {
    unsigned count, gen;
    int abort, pad;
};

// Sense by generation; release / acquire at agent scope orders the slot writes and reads across the XCDs.
// A bounded wait: past the limit the barrier sets abort and every later barrier returns at once, so the
// launch always drains. `aborted` becomes true in a workgroup that timed out or skipped a barrier for it; the
// panel kernel then writes -1 into the factor's info word, which the caller reads (the factor is not valid).
__device__ inline void grid_sync(Bar *b, unsigned nblocks, unsigned &gen, bool &aborted)
{
    __threadfence();
    __syncthreads();
    __shared__ int s_abort;
    if (threadIdx.x == 0) {
        if (!__hip_atomic_load(&b->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
            const unsigned arrived = __hip_atomic_fetch_add(&b->count, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
            if (arrived == nblocks - 1) {
                __hip_atomic_store(&b->count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_fetch_add(&b->gen, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            } else {
                long spins = 0;
                while (__hip_atomic_load(&b->gen, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) == gen) {
                    __builtin_amdgcn_s_sleep(1);
                    if (++spins > (1L << 26)) {
                        __hip_atomic_store(&b->abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        break;
                    }
                }
            }
        }
        s_abort = __hip_atomic_load(&b->abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        gen += 1;
    }
    __syncthreads();
    aborted = aborted || s_abort != 0;
}

__global__ void k_zero_ints(int *p, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void k_iota(int *p, long n)
{
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) p[i] = (int)i;
}

// ---- panel --------------------------------------------------------------------------------------------------
constexpr int NB = 128;          // panel width
constexpr int PT = 256;          // panel threads

template <typename T> struct Slot {
    double val;
    int row, pad;
    T v[NB];
};

// argmax of |Re| + |Im| over (val, row) pairs: larger value, then smaller row
__device__ inline void better(double &v, int &r, double v2, int r2)
{
    if (v2 > v || (v2 == v && r2 < r && r2 >= 0) || (r < 0 && r2 >= 0)) { v = v2; r = r2; }
}

__device__ inline void block_argmax(double &v, int &r, double *sv, int *sr)
{
    for (int o = 32; o > 0; o >>= 1) {
        const double v2 = __shfl_xor(v, o);
        const int r2 = __shfl_xor(r, o);
        better(v, r, v2, r2);
    }
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) { sv[wv] = v; sr[wv] = r; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < PT / 64; ++k) better(sv[0], sr[0], sv[k], sr[k]);
    }
    __syncthreads();
    v = sv[0]; r = sr[0];
    __syncthreads();
}

// Slab of workgroup g: global rows [r0, r0 + rn), panel columns [j0, j0 + jb), column-major in LDS (S[c * R + r]).
template <typename T>
__global__ __launch_bounds__(PT) void k_panel(T *A, long lda, long n, long j0, int jb, int R, int *ipiv, int *info,
                                              Slot<T> *slots, T *diag, Bar *bar)
{
    extern __shared__ char smem_raw[];
    T *S = (T *)smem_raw;
    __shared__ T urow[NB], drow[NB];
    __shared__ double sv[PT / 64];
    __shared__ int sr[PT / 64];
    __shared__ int piv_row;
    const unsigned G = gridDim.x;
    const int g = blockIdx.x, tid = threadIdx.x;
    const long r0 = j0 + (long)g * R;
    const int rn = (int)std::max(0L, std::min((long)R, n - r0));
    unsigned gen = 0;
    bool aborted = false;
    for (int idx = tid; idx < rn * jb; idx += PT) {
        const int c = idx / rn, r = idx % rn;
        S[c * R + r] = A[(j0 + c) * lda + r0 + r];
    }
    __syncthreads();
    // candidates of column k: rows >= j0 + k of my slab; publish (val, row, row values) in slots[buf][g], and the
    // diagonal row j0 + k in diag[buf] when it is mine
    auto publish = [&](int k, int buf) {
        double v = -1.0;
        int rr = -1;
        const long first = j0 + k;
        for (int r = tid; r < rn; r += PT)
            if (r0 + r >= first) better(v, rr, cabs1(S[k * R + r]), (int)(r0 + r));
        block_argmax(v, rr, sv, sr);
        Slot<T> *sl = slots + (size_t)buf * G + g;
        if (tid == 0) { sl->val = v; sl->row = rr; }
        if (rr >= 0)
            for (int c = tid; c < jb; c += PT) sl->v[c] = S[c * R + (rr - r0)];
        if (first >= r0 && first < r0 + rn)
            for (int c = tid; c < jb; c += PT) diag[(size_t)buf * NB + c] = S[c * R + (first - r0)];
    };
    publish(0, 0);
    grid_sync(bar, G, gen, aborted);
    for (int k = 0; k < jb; ++k) {
        const int buf = k & 1;
        const long dr = j0 + k;
        // the pivot: the best of the published candidates (every workgroup reads the same ones)
        if (tid < 64) {
            double v = -1.0;
            int rr = -1;
            for (unsigned q = tid; q < G; q += 64) {
                const Slot<T> *sl = slots + (size_t)buf * G + q;
                better(v, rr, sl->val, sl->row);
            }
            for (int o = 32; o > 0; o >>= 1) {
                const double v2 = __shfl_xor(v, o);
                const int r2 = __shfl_xor(rr, o);
                better(v, rr, v2, r2);
            }
            if (tid == 0) piv_row = rr < 0 ? (int)dr : rr;
        }
        __syncthreads();
        const int p = piv_row;
        const int gp = (int)((p - j0) / R);
        for (int c = tid; c < jb; c += PT) {
            urow[c] = slots[(size_t)buf * G + gp].v[c];
            drow[c] = diag[(size_t)buf * NB + c];
        }
        if (g == 0 && tid == 0) ipiv[dr] = p;
        __syncthreads();
        if (p != dr) {
            if (p >= r0 && p < r0 + rn)
                for (int c = tid; c < jb; c += PT) S[c * R + (p - r0)] = drow[c];
            if (dr >= r0 && dr < r0 + rn)
                for (int c = tid; c < jb; c += PT) S[c * R + (dr - r0)] = urow[c];
        }
        __syncthreads();
        const T pv = urow[k];
        const bool zero = pv.x == 0 && pv.y == 0;
        if (zero && g == 0 && tid == 0 && info && *info == 0) *info = (int)dr + 1;
        const T inv = zero ? CX<T>::make(0, 0) : trecip(pv);
        // multipliers, then the rank-1 update of the rest of the slab's panel columns
        const int rbeg = (int)std::max(0L, std::min((long)rn, dr + 1 - r0));
        if (!zero)
            for (int r = rbeg + tid; r < rn; r += PT) S[k * R + r] = tmul(S[k * R + r], inv);
        __syncthreads();
        const int nr = rn - rbeg, ncol = jb - k - 1;
        for (int idx = tid; idx < nr * ncol; idx += PT) {
            const int c = k + 1 + idx / nr, r = rbeg + idx % nr;
            S[c * R + r] = tsub(S[c * R + r], tmul(S[k * R + r], urow[c]));
        }
        __syncthreads();
        if (k + 1 < jb) {
            publish(k + 1, buf ^ 1);
            grid_sync(bar, G, gen, aborted);
        }
    }
    for (int idx = tid; idx < rn * jb; idx += PT) {
        const int c = idx / rn, r = idx % rn;
        A[(j0 + c) * lda + r0 + r] = S[c * R + r];
    }
    if (aborted && tid == 0 && info) __hip_atomic_exchange(info, -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// the panel's interchanges on columns [0, j0) and [j0 + jb, n): one thread a column, in order
template <typename T>
__global__ void k_laswp(T *A, long lda, long n, long j0, int jb, const int *ipiv)
{
    const long t = blockIdx.x * (long)blockDim.x + threadIdx.x;
    const long nleft = j0, nright = n - j0 - jb;
    if (t >= nleft + nright) return;
    const long c = t < nleft ? t : j0 + jb + (t - nleft);
    T *col = A + c * lda;
    for (int k = 0; k < jb; ++k) {
        const long r = j0 + k, p = ipiv[r];
        if (p != r) {
            const T a = col[r];
            col[r] = col[p];
            col[p] = a;
        }
    }
}

// U12 = L11^-1 A12 of the partial-pivoting panels: rows [j0, j0 + jb), columns [c0, n); TC columns a workgroup, the block
// in LDS, L11 read from memory at each step.
constexpr int TC = 16;
template <typename T>
__global__ __launch_bounds__(256) void k_trsm(T *A, long lda, long n, long j0, int jb, long c0)
{
    __shared__ T X[NB][TC + 1];
    const long cb = c0 + (long)blockIdx.x * TC;
    const int nc = (int)std::min((long)TC, n - cb);
    const int tid = threadIdx.x;
    const T *L = A + j0 * lda + j0;          // L11[i][k] = L[k * lda + i]
    for (int idx = tid; idx < jb * TC; idx += 256) {
        const int c = idx / jb, r = idx % jb;
        if (c < nc) X[r][c] = A[(cb + c) * lda + j0 + r];
    }
    __syncthreads();
    for (int k = 0; k < jb - 1; ++k) {
        const int nr = jb - k - 1;
        for (int idx = tid; idx < nr * TC; idx += 256) {
            const int c = idx % TC, i = k + 1 + idx / TC;
            if (c < nc) X[i][c] = tsub(X[i][c], tmul(L[(long)k * lda + i], X[k][c]));
        }
        __syncthreads();
    }
    for (int idx = tid; idx < jb * TC; idx += 256) {
        const int c = idx / jb, r = idx % jb;
        if (c < nc) A[(cb + c) * lda + j0 + r] = X[r][c];
    }
}

// ---- C -= A B on the matrix cores ---------------------------------------------------------------------------
// C (M x N), A (M x K), B (K x N), column-major, complex; K a multiple of KS. Workgroup tile 64 x 64, eight waves of 32 x
// 16, each 2 blocks of 16 x 16 with a real and an imaginary accumulator. The MFMA's first operand is B (its rows are
// C's columns), its second A, so a lane's outputs run down C's columns (coalesced stores). At K = 64 an update moves as
// much time's worth of C as it computes (c128: 32 B an entry for 512 flops), so the two have to overlap: a tile's C is
// asked for first and met last, the stages of A and B alternate between two LDS buffers with one barrier a stage, and
// the tiles are small and the waves narrow so that four and more a SIMD are at different points of theirs. Loads past
// the matrix read its last row or column instead of branching (what they feed is never stored). Workgroups are dealt to
// the eight XCDs round robin; XCD x takes the x-th run of tiles, columns of tiles in order, so its L2 keeps its part of
// B and the rows of A it meets. Measured at M = 7735, K = 64: 77 -> 89 TFLOP/s (complex64), 37 -> 52 (complex128); tiles of
// 128 x 64 and 128 x 128, 16-column stages and a persistent grid keeping A's tile measured slower (47 to 87, 30 to 51).
constexpr int GM = 64, GN = 64, GK = 8, GT = 512;
constexpr int GWR = 2, GWC = 4;                 // waves down and across a tile

template <typename T, typename AC = T, int KS = GK>
__device__ __forceinline__ void gemm_body(T *C, long ldc, const T *A, long lda, const T *B, long ldb, long M, long N,
                                          long K, long bx, long by)
{
    typedef typename CX<AC>::R R;           // the matrix cores' type: products and sums in it, one rounding to T
    typedef typename CX<T>::R TR;
    typedef typename CX<AC>::acc4 acc4;
    constexpr int LA = GM * KS / GT, LB = KS * GN / GT;     // a thread's elements of A and of B a stage
    constexpr int FA = GM / GWR / 16, FB = GN / GWC / 16;   // a wave's 16 x 16 blocks
    __shared__ T As[2][KS][GM];         // As[s][p][i] = A[i][p]
    __shared__ T Bs[2][KS][GN + 1];     // Bs[s][p][j] = B[p][j]
    const long m0 = bx * GM, n0 = by * GN;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int wm = (wv % GWR) * (GM / GWR), wn = (wv / GWR) * (GN / GWC);     // wave tile origin in the workgroup tile
    const int li = lane & 15, kk = lane >> 4, part = kk & 1, ph = kk >> 1;
    // (complex values held in registers are kept as separate real and imaginary arrays: an array of the vector type
    // goes to scratch memory for complex128)
    TR rax[LA], ray[LA], rbx[LB], rby[LB];
    auto fetch = [&](long k0) __attribute__((always_inline)) {
#pragma unroll
        for (int it = 0; it < LA; ++it) {
            const int idx = tid + it * GT, i = idx % GM, p = idx / GM;
            const T v = A[(k0 + p) * lda + std::min(m0 + i, M - 1)];
            rax[it] = v.x; ray[it] = v.y;
        }
#pragma unroll
        for (int it = 0; it < LB; ++it) {
            const int idx = tid + it * GT, p = idx % KS, j = idx / KS;
            const T v = B[std::min(n0 + j, N - 1) * ldb + k0 + p];
            rbx[it] = v.x; rby[it] = v.y;
        }
    };
    auto stage = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int it = 0; it < LA; ++it) {
            const int idx = tid + it * GT;
            As[s][idx / GM][idx % GM] = CX<T>::make(rax[it], ray[it]);
        }
#pragma unroll
        for (int it = 0; it < LB; ++it) {
            const int idx = tid + it * GT;
            Bs[s][idx % KS][idx / KS] = CX<T>::make(rbx[it], rby[it]);
        }
    };
    // lane (li, kk), register r: C row m0 + wm + a*16 + li, column n0 + wn + b*16 + out_row(kk, r)
    auto row_of = [&](int a) { return m0 + wm + a * 16 + li; };
    auto col_of = [&](int b, int r) { return n0 + wn + b * 16 + CX<AC>::out_row(kk, r); };
    fetch(0);
    TR cx[FB][FA][4], cy[FB][FA][4];
#pragma unroll
    for (int b = 0; b < FB; ++b)
#pragma unroll
        for (int a = 0; a < FA; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const T v = C[std::min(col_of(b, r), N - 1) * ldc + std::min(row_of(a), M - 1)];
                cx[b][a][r] = v.x; cy[b][a][r] = v.y;
            }
    acc4 cr[FB][FA], ci[FB][FA];
#pragma unroll
    for (int b = 0; b < FB; ++b)
#pragma unroll
        for (int a = 0; a < FA; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r) { cr[b][a][r] = 0; ci[b][a][r] = 0; }
    stage(0);
    __syncthreads();
    int s = 0;
    for (long k0 = 0; k0 < K; k0 += KS, s ^= 1) {
        const bool more = k0 + KS < K;
        if (more) fetch(k0 + KS);
#pragma unroll
        for (int ks = 0; ks < KS / 2; ++ks) {
            const int p = 2 * ks + ph;
            R av[FA], br[FB], bi[FB];
#pragma unroll
            for (int a = 0; a < FA; ++a) av[a] = (R)((const TR *)&As[s][p][wm + a * 16 + li])[part];
#pragma unroll
            for (int b = 0; b < FB; ++b) {
                const T y = Bs[s][p][wn + b * 16 + li];
                br[b] = (R)(part ? -y.y : y.x);
                bi[b] = (R)(part ? y.x : y.y);
            }
#pragma unroll
            for (int b = 0; b < FB; ++b)
#pragma unroll
                for (int a = 0; a < FA; ++a) {
                    cr[b][a] = CX<AC>::mfma(br[b], av[a], cr[b][a]);
                    ci[b][a] = CX<AC>::mfma(bi[b], av[a], ci[b][a]);
                }
        }
        if (more) stage(s ^ 1);
        __syncthreads();
    }
    const bool whole = m0 + GM <= M && n0 + GN <= N;
#pragma unroll
    for (int b = 0; b < FB; ++b)
#pragma unroll
        for (int a = 0; a < FA; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (whole || (row_of(a) < M && col_of(b, r) < N))
                    C[col_of(b, r) * ldc + row_of(a)] = CX<T>::make((TR)((R)cx[b][a][r] - cr[b][a][r]),
                                                                    (TR)((R)cy[b][a][r] - ci[b][a][r]));
}

inline unsigned gemm_grid(long M, long N)
{
    const long t = ((M + GM - 1) / GM) * ((N + GN - 1) / GN);
    return (unsigned)(8 * ((t + 7) / 8));
}

// one workgroup a tile of gemm_grid(M, N); the XCD (workgroup i runs on XCD i % 8) takes its run of the tiles
template <typename T, typename AC = T, int KS = GK>
__global__ __launch_bounds__(GT) void k_gemm(T *C, long ldc, const T *A, long lda, const T *B, long ldb, long M,
                                             long N, long K)
{
    const long tm = (M + GM - 1) / GM, t = (blockIdx.x & 7) * (long)(gridDim.x >> 3) + (blockIdx.x >> 3);
    if (t >= tm * ((N + GN - 1) / GN)) return;
    gemm_body<T, AC, KS>(C, ldc, A, lda, B, ldb, M, N, K, t % tm, t / tm);
}

// The depth of the K stages of the tournament LU's trailing update (8, 16 or 32: the number of columns of L21 and
// rows of U12 staged in LDS between two barriers), chosen at run time by m25x_lu_set_gemm_stage (an autotuner
// times the choices); 8 until set.
std::atomic<int> g_gemm_stage{8};
// The complex64 trailing update's matrix cores: 1 FP32 (the default: v_mfma_f32_16x16x4f32, FP32 accumulation, twice
// the FP64 peak rate), 0 FP64 (v_mfma_f64_16x16x4f64, products and sums in FP64, one rounding to FP32 per update:
// a smaller backward error); m25x_lu_set_update_precision. complex128 always updates in FP64.
std::atomic<int> g_update_fp32{1};

template <typename T, typename AC>
void launch_update_ac(hipStream_t s, T *C, long ldc, const T *A, long lda, const T *B, long ldb, long M, long N, long K)
{
    const dim3 grid(gemm_grid(M, N));
    switch (g_gemm_stage.load(std::memory_order_relaxed)) {
    case 16: hipLaunchKernelGGL((k_gemm<T, AC, 16>), grid, dim3(GT), 0, s, C, ldc, A, lda, B, ldb, M, N, K); break;
    case 32: hipLaunchKernelGGL((k_gemm<T, AC, 32>), grid, dim3(GT), 0, s, C, ldc, A, lda, B, ldb, M, N, K); break;
    default: hipLaunchKernelGGL((k_gemm<T, AC, 8>), grid, dim3(GT), 0, s, C, ldc, A, lda, B, ldb, M, N, K);
    }
}

template <typename T>
void launch_update(hipStream_t s, T *C, long ldc, const T *A, long lda, const T *B, long ldb, long M, long N, long K)
{
    if constexpr (sizeof(T) == 8) {
        if (g_update_fp32.load(std::memory_order_relaxed)) {
            launch_update_ac<T, float2>(s, C, ldc, A, lda, B, ldb, M, N, K);
            return;
        }
    }
    launch_update_ac<T, double2>(s, C, ldc, A, lda, B, ldb, M, N, K);
}

// ---- the interchanges as a permutation: perm = the swaps of ipiv applied in order to 0..n-1 ------------------
__global__ void k_perm(const int *ipiv, long n, int *perm)
{
    // one workgroup: identity in parallel, then the swaps in order by one thread, ipiv read 8 at a time (the
    // loads are independent of the swaps; most pivots are on the diagonal)
    for (long i = threadIdx.x; i < n; i += blockDim.x) perm[i] = (int)i;
    __threadfence_block();
    __syncthreads();
    if (threadIdx.x == 0) {
        for (long i0 = 0; i0 < n; i0 += 8) {
            int pv[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) pv[u] = i0 + u < n ? ipiv[i0 + u] : (int)(i0 + u);
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const long i = i0 + u;
                const int p = pv[u];
                if (i < n && p != i) {
                    const int t = perm[i];
                    perm[i] = perm[p];
                    perm[p] = t;
                }
            }
        }
    }
}

// rows of a block of the triangular solves, and their most right-hand sides
constexpr int SB = 64;
constexpr int MAXRHS = 8;

// A tournament panel's L21 = A21 U11^-1 (x U11 = a for each row a below the panel) and U12 = L11^-1 A12 (L11 x = a for
// each column a right of it) by substitution: 64 unknowns a vector, the triangle (from top) in LDS. Sixteen lanes (a DPP
// row) share a vector, lane l holding its elements l, l + 16, l + 32, l + 48; step k broadcasts the finished element k
// among them (row_newbcast) and every lane subtracts its multiple from the later elements. What bounds it is how many
// lanes work and the steps' latency: with a row a thread L21 kept 120 of the chip's 1024 SIMDs busy at N = 7799, and U12
// passed 63 barriers. TRI_V vectors a lane, 32 a workgroup of 256 threads, cover the chip and give a step independent
// work. Measured, both blocks of a panel at N = 7799: 78 us (complex64), 99 us (complex128) before; 11.8 and 15.4 us so.
constexpr int TRI_V = 2, TRI_N = 16 * TRI_V;          // vectors a workgroup
template <int N> __device__ __forceinline__ float row_bcast(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + N, 0xF, 0xF, true));
}
template <int N> __device__ __forceinline__ double row_bcast(double v)
{
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)b, 0x150 + N, 0xF, 0xF, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x150 + N, 0xF, 0xF, true);
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

// UPPER: rows [r0 + 32 bx, ...) of L21 (m rows from r0 = j0 + TW); else columns of U12 (the same m from r0)
template <typename T, bool UPPER>
__device__ __forceinline__ void tri_vectors(T *A, long lda, long j0, long m, const T *top, long bx, T (*M)[TW + 1], T *rd)
{
    const int tid = threadIdx.x, l16 = tid & 15;
    const long r0 = j0 + TW, v0 = bx * TRI_N + (tid >> 6) * (4 * TRI_V) + ((tid >> 4) & 3);
    const long es = UPPER ? lda : 1, vs = UPPER ? 1 : lda;         // steps between elements and between vectors
    T *base = A + (UPPER ? j0 * lda + r0 : r0 * lda + j0);
    T v[TW * TW / 256];                               // every load in flight before the first store
#pragma unroll
    for (int u = 0; u < TW * TW / 256; ++u) v[u] = top[tid + u * 256];
    T a[TRI_V][4];
#pragma unroll
    for (int q = 0; q < TRI_V; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) a[q][i] = base[std::min(v0 + 4 * q, m - 1) * vs + (l16 + 16 * i) * es];
    const T zero = CX<T>::make(0, 0);
    if (UPPER && tid < TW) rd[tid] = trecip(top[tid * (TW + 1)]);
#pragma unroll
    for (int u = 0; u < TW * TW / 256; ++u) {         // top: column e / 64, row e % 64; M[k][c]: element c's multiple of
        const int e = tid + u * 256, c = e / TW, i = e % TW;      // element k, zero for c <= k
        if (UPPER) M[i][c] = csel(i < c, v[u], zero);
        else M[c][i] = csel(i > c, v[u], zero);
    }
    __syncthreads();
    auto step = [&](auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value, ik = k / 16;
        T x[TRI_V];
#pragma unroll
        for (int q = 0; q < TRI_V; ++q) {
            x[q] = CX<T>::make(row_bcast<k % 16>(a[q][ik].x), row_bcast<k % 16>(a[q][ik].y));
            if (UPPER) x[q] = tmul(x[q], rd[k]);
        }
#pragma unroll
        for (int i = ik; i < 4; ++i) {
            const T mk = M[k][l16 + 16 * i];
#pragma unroll
            for (int q = 0; q < TRI_V; ++q) a[q][i] = tfms(a[q][i], x[q], mk);
        }
    };
    Unroll<0, TW - 1>::run(step);
#pragma unroll
    for (int q = 0; q < TRI_V; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (v0 + 4 * q < m)
                base[(v0 + 4 * q) * vs + (l16 + 16 * i) * es] = UPPER ? tmul(a[q][i], rd[l16 + 16 * i]) : a[q][i];
}

// workgroup bx of 2 nb21: the first half L21, the other U12
template <typename T>
__device__ __forceinline__ void tri_body(T *A, long lda, long j0, long m, const T *top, long bx, long nb21)
{
    __shared__ T M[TW][TW + 1];
    __shared__ T rd[TW];
    if (bx < nb21) tri_vectors<T, true>(A, lda, j0, m, top, bx, M, rd);
    else tri_vectors<T, false>(A, lda, j0, m, top, bx - nb21, M, rd);
}

template <typename T>
__global__ __launch_bounds__(256) void k_tri(T *A, long lda, long j0, long m, const T *top)
{
    tri_body<T>(A, lda, j0, m, top, blockIdx.x, (long)gridDim.x / 2);
}

// The panel's row moves on columns [c0, c0 + nc): a column per 128 threads, every source read before any write;
// the panel's own columns [j0, j0 + jb) then take the root's L11 \ U11 in rows [j0, j0 + jb). With perm, one more
// workgroup moves the entries of the row permutation (position -> original row) the same way.
template <typename T>
__device__ __forceinline__ void apply_moves_body(T *A, long lda, long c0, long nc, const int *pairs, long j0, int jb,
                                                 const T *top, int *perm, long bx, long perm_block)
{
    const int t = threadIdx.x & 127, h = threadIdx.x >> 7;
    const int np = pairs[0];
    const int dst = t < np ? pairs[1 + 2 * t] : 0, src = t < np ? pairs[2 + 2 * t] : 0;
    if (perm && bx == perm_block) {                 // the extra workgroup: the same moves on the row permutation
        int v = 0;
        if (h == 0 && t < np) v = perm[src];
        __syncthreads();
        if (h == 0 && t < np) perm[dst] = v;
        return;
    }
    T v[4];                                         // the workgroup's 8 columns, two at a time: all read first
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const long cb = bx * 8 + 2 * u;
        v[u] = ldz(cb + h < nc && t < np, A + (c0 + cb + h) * lda + src);
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const long cb = bx * 8 + 2 * u, c = c0 + cb + h;
        if (cb + h < nc && t < np) A[c * lda + dst] = v[u];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const long cb = bx * 8 + 2 * u, c = c0 + cb + h;
        if (cb + h < nc && c >= j0 && c < j0 + jb)
            for (int i = t; i < jb; i += 128) A[c * lda + j0 + i] = top[(c - j0) * TW + i];
    }
}

// grid: blocks(nc, 8) workgroups of columns, and with perm one more (the last) for the permutation
template <typename T>
__global__ __launch_bounds__(256) void k_apply_moves(T *A, long lda, long c0, long nc, const int *pairs, long j0,
                                                     int jb, const T *top, int *perm)
{
    apply_moves_body<T>(A, lda, c0, nc, pairs, j0, jb, top, perm, blockIdx.x, (long)gridDim.x - 1);
}

__device__ inline double readlane_d(double v, int l)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ inline double2 readlane_c(double2 v, int l) { return make_double2(readlane_d(v.x, l), readlane_d(v.y, l)); }

// ---- values that carry their own ready mark ----------------------------------------------------------------
// The solves hand results between workgroups through buffers filled beforehand with all-ones 64-bit words (a NaN
// pattern no arithmetic produces): every 64-bit word is written and read with single-copy atomic accesses at
// device scope, so a reader that finds no all-ones word in a value has the value itself, with no flag and no
// second round trip. A computed word that happens to be all ones is written as the canonical NaN instead.
typedef unsigned long long u64;
constexpr u64 UNSET = ~0ull;

__device__ inline u64 mark_safe(u64 w, u64 nan) { return w == UNSET ? nan : w; }
__device__ inline void put(float2 *p, float2 v)
{
    const u64 w = ((u64)__float_as_uint(v.y) << 32) | __float_as_uint(v.x);
    __hip_atomic_store((u64 *)p, mark_safe(w, 0x7fc000007fc00000ull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void put(double2 *p, double2 v)
{
    u64 *q = (u64 *)p;
    __hip_atomic_store(q, mark_safe((u64)__double_as_longlong(v.x), 0x7ff8000000000000ull), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(q + 1, mark_safe((u64)__double_as_longlong(v.y), 0x7ff8000000000000ull), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
// the value at p (all-ones words if it has not been written yet), and whether it has been written
__device__ inline float2 fetch(const float2 *p)
{
    const u64 w = __hip_atomic_load((u64 *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return make_float2(__uint_as_float((unsigned)w), __uint_as_float((unsigned)(w >> 32)));
}
__device__ inline double2 fetch(const double2 *p)
{
    const u64 a = __hip_atomic_load((u64 *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const u64 b = __hip_atomic_load((u64 *)p + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return make_double2(__longlong_as_double((long long)a), __longlong_as_double((long long)b));
}
__device__ inline bool is_set(float2 v) { return (__float_as_uint(v.x) & __float_as_uint(v.y)) != ~0u; }
__device__ inline bool is_set(double2 v)
{
    return (u64)__double_as_longlong(v.x) != UNSET && (u64)__double_as_longlong(v.y) != UNSET;
}
template <typename T> __device__ inline bool take(const T *p, T &v)
{
    v = fetch(p);
    return is_set(v);
}
__device__ inline bool wave_all(bool c) { return __builtin_amdgcn_ballot_w64(!c) == 0; }

// ---- the triangular solves ---------------------------------------------------------------------------------
// One launch solves both triangles for all right-hand sides, two to a chain: workgroup q of a chain's pass owns the q-th
// 64-row diagonal block in solve order and hands its solution to the workgroups after it; the second pass's workgroups
// take the first one's solution as their right-hand side. The chains of a call run side by side (a solve is bound by the
// latency from block to block, not by the chip), the workgroups of one block in one XCD so that its L2 serves the
// block's rows to all of them, and the second pass's workgroups prepare their blocks while the first pass runs.
//
// A workgroup waits only for blocks of its chain before its own, and it begins to wait for them only once workgroups that
// have started answer for all of those (gate); where one stays away it does that one's block first. So as soon as any
// workgroup of a chain runs, the chain's first unfinished block is being worked on by one that waits for nothing, and
// every launch makes progress with any number of its workgroups resident and whatever else is on the device. The order
// of the numbers alone does not give that: each XCD starts its own workgroups in order, but nothing holds the XCDs in
// step, and of two solves at once on two streams (a complex64 workgroup has a CU to itself) each could fill one XCD with
// workgroups that wait for a block the other one keeps out. (Numbers drawn from a counter at the start give it too, but
// an XCD's workgroups start in a burst and draw neighbouring blocks: complex128 solves took 5 to 9 % longer.)
//
// y travels as self-marking values (put / take) in dst, chain after chain, the pair of a row side by side: a reader
// spins on the values themselves, every lane on its own when the block is one of the two before its own (the chain
// waits on it), one lane with growing naps first otherwise.
constexpr int TB = 512;                  // threads of a solve workgroup: 8 waves
constexpr int NWV = TB / 64;
constexpr int TE = SB * SB / TB;         // entries of a 64 x 64 tile a thread takes: 8
constexpr int CR = 2;                    // right-hand sides of a chain

template <typename T> struct Tri {       // one chain's solve of one triangle
    const T *LU;
    long lda, n;
    const T *src;                        // right-hand side: row i at src[(sperm ? sperm[i] : i) * lds + r]
    long lds;
    const int *sperm;
    bool wait;                           // src holds self-marking values
    T *dst;                              // n x CR solution values, UNSET words before the launch
    T *out;                              // if given, the solution again: row i at out[(operm ? operm[i] : i) * ldo + r]
    long ldo;
    const int *operm;
    int kc;                              // right-hand sides in use (1 or 2; the other one solves for zero)
    bool fwd, unit;                      // rows in ascending order (else descending); unit diagonal
    int *abort;                          // raised if a wait exceeds its bound (the result is then garbage, not a hang)
};

// workgroup -> (pass, block in solve order, chain): the chains of block q are 8 apart, in q's XCD
struct ChainPos {
    int pass, q, chain;
};
__host__ __device__ inline int chain_wgs(int nb, int nchain) { return (nb + 7) / 8 * 8 * nchain; }      // of a pass
__device__ inline ChainPos chain_pos(int wg, int nb, int nchain)
{
    const int per = chain_wgs(nb, nchain), pass = wg / per, w = wg - pass * per, t = w / 8;
    return ChainPos{pass, t / nchain * 8 + w % 8, t % nchain};
}

// The blocks of a chain, both passes in order, a bit each: those whose workgroup has started, or that another workgroup
// does for it, and those that a workgroup has taken to do, which only one can.
__host__ __device__ inline int held_words(int nb) { return (2 * nb + 63) / 64; }
struct Held {
    u64 *started, *taken;
};
__device__ inline Held held_of(u64 *held, int chain, int nb)
{
    const int w = held_words(nb);
    return Held{held + 2 * chain * w, held + (2 * chain + 1) * w};
}
__device__ inline void start_block(const Held &h, int i)
{
    __hip_atomic_fetch_or(h.started + (i >> 6), 1ull << (i & 63), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline bool take_block(const Held &h, int i)
{
    const u64 bit = 1ull << (i & 63);
    return !(__hip_atomic_fetch_or(h.taken + (i >> 6), bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bit);
}
// the first block before `end` that has not started, or -1 (a whole wave calls)
__device__ inline int first_missing(const Held &h, int end)
{
    for (int b0 = 0; b0 * 64 < end; b0 += 64) {
        const int b = b0 + (threadIdx.x & 63), left = end - b * 64;
        const u64 need = left <= 0 ? 0 : left >= 64 ? ~0ull : (1ull << left) - 1;
        u64 miss = 0;
        if (need) miss = need & ~__hip_atomic_load(h.started + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const u64 any = __builtin_amdgcn_ballot_w64(miss != 0);
        if (any) {
            const int l = __builtin_ctzll(any);
            const u64 m = (u64)(unsigned)__builtin_amdgcn_readlane((int)(miss >> 32), l) << 32 |
                          (unsigned)__builtin_amdgcn_readlane((int)miss, l);
            return (b0 + l) * 64 + __builtin_ctzll(m);
        }
    }
    return -1;
}
// The block that the workgroup with block `own` goes on with: its own once all before it have started, the first missing
// one where it has waited for that long enough, -1 where another workgroup has taken its own. All threads call. The
// workgroups of an empty chip start within a third of a us of each other and ask when their blocks are prepared; later
// ones start as an XCD's slots come free, up to 40 us apart (8 blocks of 3.3 us and more). The patience is ten times
// that: a block that another workgroup does delays the chain.
constexpr int GATE_POLLS = 400;          // about a us each
__device__ __forceinline__ int gate(const Held &h, int own)
{
    __shared__ int next;
    if (threadIdx.x < 64) {
        int got = 0, i = first_missing(h, own);
        for (int polls = 0; i >= 0; ++polls) {
            if (polls >= GATE_POLLS) {
                if (threadIdx.x == 0 && (got = take_block(h, i))) start_block(h, i);
                if (__builtin_amdgcn_readfirstlane(got)) break;
            }
            __builtin_amdgcn_s_sleep(8);
            i = first_missing(h, own);
        }
        if (threadIdx.x == 0) next = i >= 0 ? i : take_block(h, own) ? own : -1;
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(next);
}

// A workgroup's turn at block i of its chain (both passes in order; `own` is its own)
struct Turn {
    Held h;
    int own, i, next;
    // Once before the first wait for another block: whether to go on with block i. (A block taken to be done for another
    // workgroup has none missing before it.)
    __device__ __forceinline__ bool go()
    {
        next = i == own ? gate(h, own) : i;
        return next == i;
    }
};

template <typename T> __device__ inline void to_out(const Tri<T> &c, long gi, long go, int r, T v)
{
    put(c.dst + gi * CR + r, v);
    if (c.out && r < c.kc) c.out[go * c.ldo + r] = v;
}

// Polls until the condition holds in every lane of the wave (ok, then what attempt() returns), or the bound is reached
// (abort raised).
template <bool NAP, class Try> __device__ __forceinline__ void wave_wait(bool ok, int *abort, Try &&attempt)
{
    long spins = 0;
    while (!wave_all(ok)) {
        if (NAP) __builtin_amdgcn_s_sleep(1);
        if (++spins > (1L << 22)) {
            __hip_atomic_store(abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
        }
        if (!ok) ok = attempt();
    }
}
// d blocks from the chain one lane watches a value, with naps that grow to d / 16 of a us: every later workgroup reads
// the chain's newest values, and tight polls of all of them on one line would hold up the one that the chain waits for
template <typename T> __device__ __forceinline__ void nap_wait(const T *w0, int d, int *abort)
{
    T v;
    long spins = 0;
    const int most = std::min(d, 64);
    int nap = 1 + most / 8;
    while (!take(w0, v)) {
        for (int z = 0; z < nap; ++z) __builtin_amdgcn_s_sleep(2);
        nap = std::min(2 * nap, most);
        if (++spins > (1L << 22)) {
            __hip_atomic_store(abort, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
        }
    }
}
// row gi of the chain's right-hand sides (every lane of the wave calls)
template <typename T> __device__ __forceinline__ void rhs_row(const Tri<T> &c, long gi, T (&b)[CR])
{
    if (c.wait) {
        const T *p = c.src + gi * CR;
        auto attempt = [&]() {
            const bool a0 = take(p, b[0]), a1 = take(p + 1, b[1]);
            return a0 && a1;
        };
        const bool ok = attempt();
        if (!wave_all(ok)) {
            if ((threadIdx.x & 63) == 0) nap_wait(p, 64, c.abort);
            wave_wait<true>(ok, c.abort, attempt);
        }
        return;
    }
    const T *p = c.src + (c.sperm ? (long)c.sperm[gi] : gi) * c.lds;
    b[0] = p[0];
    b[1] = csel(c.kc > 1, p[c.kc > 1 ? 1 : 0], CX<T>::make(0, 0));
}

// right-hand side r of rows g0 and g1
template <typename T> __device__ __forceinline__ void rhs_pair(const Tri<T> &c, long g0, long g1, int r, T (&b)[2])
{
    if (c.wait) {
        const T *p0 = c.src + g0 * CR + r, *p1 = c.src + g1 * CR + r;
        auto attempt = [&]() {
            const bool a0 = take(p0, b[0]), a1 = take(p1, b[1]);
            return a0 && a1;
        };
        const bool ok = attempt();
        if (!wave_all(ok)) {
            if ((threadIdx.x & 63) == 0) nap_wait(p0, 64, c.abort);
            wave_wait<true>(ok, c.abort, attempt);
        }
        return;
    }
    const int rr = r < c.kc ? r : 0;
    const T zero = CX<T>::make(0, 0);
    b[0] = csel(r < c.kc, c.src[(c.sperm ? (long)c.sperm[g0] : g0) * c.lds + rr], zero);
    b[1] = csel(r < c.kc, c.src[(c.sperm ? (long)c.sperm[g1] : g1) * c.lds + rr], zero);
}

// sums within groups of lanes by DPP moves: quad_perm [1,0,3,2] (0xB1), quad_perm [2,3,0,1] (0x4E); and over the halves and quarters of a wave by lane swaps
template <int CTRL> __device__ __forceinline__ float dpp_of(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
template <int CTRL> __device__ __forceinline__ double dpp_of(double v)
{
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, true);
    const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | lo);
}
__device__ __forceinline__ float swap32_add(float a, float b)     // lanes 0-31: a over both halves; 32-63: b
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float swap16_add(float a, float b)     // even rows of 16 lanes: a over the pair; odd: b
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ double join(unsigned lo, unsigned hi) { return __longlong_as_double(((long long)hi << 32) | lo); }
__device__ __forceinline__ double swap32_add(double a, double b)
{
    const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    return join(lo[0], hi[0]) + join(lo[1], hi[1]);
}
__device__ __forceinline__ double swap16_add(double a, double b)
{
    const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    return join(lo[0], hi[0]) + join(lo[1], hi[1]);
}

// ---- the blocks before a workgroup's own: sum_a Op_qa y_a ----
// Lane (rl, cq) of wave wv takes rows row(u) and columns 8 wv + 2 cq + v of a 64 x 64 tile, u < 4, v < 2: its loads of 16
// bytes cover whole lines in either order (row-major: 4 lanes a row; column-major: 16 lanes a column) and it polls y of
// its own two columns. (A row a lane, as the diagonal block is read, touches 64 lines a load in a row-major factor: of a
// complex128 solve at N = 7799 it took 0.4 ms.) Tiles are loaded two (complex128) or three blocks ahead of the y they
// meet.
typedef float f4u __attribute__((ext_vector_type(4), aligned(8)));    // two complex64, 8-byte aligned
template <typename T> struct Depth { static constexpr int D = 3; };
template <> struct Depth<double2> { static constexpr int D = 2; };
template <typename T> struct Tile {      // entry 2 u + v: row(u), column 2 cq + v
    typename CX<T>::R r[TE], i[TE];
    __device__ __forceinline__ void set(int e, T w)
    {
        r[e] = w.x;
        i[e] = w.y;
    }
};
// column-major complex64 rows come in pairs (a load holds two)
template <typename T, bool RM> __device__ inline int tile_row(int rl, int u)
{
    return RM || sizeof(T) == 16 ? rl + 16 * u : 2 * rl + (u & 1) + 32 * (u >> 1);
}

template <typename T, bool RM>
__device__ __forceinline__ void load_tile(Tile<T> &t, const Tri<T> &c, long r0, int m, long k0, int rl, int cq)
{
    const long gk = k0 + 2 * cq;
    const bool whole = k0 + TE <= c.n && m == SB;
    if (whole && sizeof(T) == 8) {
#pragma unroll
        for (int h = 0; h < 4; ++h) {    // row-major: two columns of row h; column-major: two rows of a column
            const T *p = RM ? c.LU + (r0 + rl + 16 * h) * c.lda + gk
                            : c.LU + (gk + (h & 1)) * c.lda + r0 + 2 * rl + 32 * (h >> 1);
            const f4u w = *(const f4u *)p;
            const int e0 = RM ? 2 * h : 4 * (h >> 1) + (h & 1), e1 = RM ? 2 * h + 1 : e0 + 2;
            t.r[e0] = w.x; t.i[e0] = w.y; t.r[e1] = w.z; t.i[e1] = w.w;
        }
        return;
    }
    // rows past the block read its last row (their sums are not used), columns past the matrix its last column (y = 0)
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            const long gi = r0 + std::min(tile_row<T, RM>(rl, u), m - 1), g = std::min(gk + v, c.n - 1);
            t.set(2 * u + v, RM ? c.LU[gi * c.lda + g] : c.LU[g * c.lda + gi]);
        }
}

// The first D tiles of the sum over blocks 0 .. nfar - 1 of the solve order.
template <typename T, bool RM, int D, class Order>
__device__ __forceinline__ void far_begin(Tile<T> (&t)[D], const Tri<T> &c, int nfar, long r0, int m, int wv, int lane,
                                          Order &&order)
{
    const int rl = RM ? lane >> 2 : lane & 15, cq = RM ? lane & 3 : lane >> 4;
#pragma unroll
    for (int d = 0; d < D; ++d)
        if (d < nfar) load_tile<T, RM>(t[d], c, r0, m, (long)order(d) * SB + wv * TE, rl, cq);
}
// o: minus the wave's part of the sum for one row a lane (re and im of the right-hand sides); returns the row. q: the
// workgroup's own place in the order (how urgent a value is).
template <typename T, bool RM, int D, class Order>
__device__ __forceinline__ int far_sum(typename CX<T>::R (&o)[2 * CR], Tile<T> (&t)[D], const Tri<T> &c, int q, int nfar,
                                       long r0, int m, int wv, int lane, Order &&order)
{
    typedef typename CX<T>::R R;
    const int rl = RM ? lane >> 2 : lane & 15, cq = RM ? lane & 3 : lane >> 4;
    const long n = c.n;
    R sr[4][CR], si[4][CR];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int r = 0; r < CR; ++r) sr[u][r] = si[u][r] = 0;
    // y of a block for this lane, (column v, right-hand side r) at 2 v + r, asked for a step ahead and before the step's
    // tile: loads return in order, and a poll behind a tile's loads would wait for them
    T yn[4];
    auto ask = [&](int p) __attribute__((always_inline)) {
        const long gk = (long)order(p) * SB + wv * TE + 2 * cq;
        bool all = true;
#pragma unroll
        for (int e = 0; e < 4; ++e) all &= take(c.dst + std::min(gk + e / 2, n - 1) * CR + e % 2, yn[e]);
        return all;
    };
    if (nfar > 0) ask(0);
    auto step = [&](int p, Tile<T> &tp) __attribute__((always_inline)) {
        const long k0 = (long)order(p) * SB + wv * TE, gk = k0 + 2 * cq;
        bool ok = true;
#pragma unroll
        for (int e = 0; e < 4; ++e) ok &= is_set(yn[e]);
        ok |= !(gk < n);
        if (!wave_all(ok)) {
            if (q - p > 2 && lane == 0 && k0 < n) nap_wait(c.dst + k0 * CR, q - p, c.abort);
            wave_wait<true>(ok, c.abort, [&]() { return ask(p); });
        }
        T y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = csel(gk + e / 2 < n, yn[e], CX<T>::make(0, 0));
        if (p + 1 < nfar) ask(p + 1);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int v = 0; v < 2; ++v)
#pragma unroll
                for (int r = 0; r < CR; ++r) {
                    const T w = tfms(CX<T>::make(sr[u][r], si[u][r]), CX<T>::make(tp.r[2 * u + v], tp.i[2 * u + v]),
                                     y[2 * v + r]);
                    sr[u][r] = w.x;
                    si[u][r] = w.y;
                }
        if (p + D < nfar) load_tile<T, RM>(tp, c, r0, m, (long)order(p + D) * SB + wv * TE, rl, cq);
    };
    for (int p = 0; p < nfar; p += D) {
#pragma unroll
        for (int d = 0; d < D; ++d)
            if (p + d < nfar) step(p + d, t[d]);
    }
    // the four lanes of a row exchange: each ends with row(cq)'s sum
#pragma unroll
    for (int e = 0; e < 2 * CR; ++e) {
        const R a0 = e & 1 ? si[0][e / 2] : sr[0][e / 2], a1 = e & 1 ? si[1][e / 2] : sr[1][e / 2],
                a2 = e & 1 ? si[2][e / 2] : sr[2][e / 2], a3 = e & 1 ? si[3][e / 2] : sr[3][e / 2];
        if (RM) {
            const bool b0 = cq & 1, b1 = cq & 2;
            const R k0 = (b0 ? a1 : a0) + dpp_of<0xB1>(b0 ? a0 : a1);
            const R k1 = (b0 ? a3 : a2) + dpp_of<0xB1>(b0 ? a2 : a3);
            o[e] = (b1 ? k1 : k0) + dpp_of<0x4E>(b1 ? k0 : k1);
        } else {
            o[e] = swap16_add(swap32_add(a0, a2), swap32_add(a1, a3));
        }
    }
    return tile_row<T, RM>(rl, cq);
}

// -- complex64 --
// The block's own triangle is inverted in FP64 when the workgroup starts, and the inverse multiplied into the tile of
// the block before it (W = inv(Op_qq) Op_q,q-1, FP64 too): a block's step is then y_q = z_q - W y_q-1, one product,
// with z_q = inv(Op_qq) (b_q - sum over a < q - 1 of Op_qa y_a) formed by the other half of the waves while y_q-1 is
// still on its way. Substitution needs 64 dependent steps instead, 1.4 us at 52 cycles (a broadcast and two dependent
// multiply-adds): the block's step went from 3.0 to 1.4 us, of which the way from one workgroup's store to the next one's
// sight of it is about 1.0 (0.54 with one line and nothing else on the way; it grows with the lines a poll asks for, but
// passing them on in LDS costs as much), and a solve of N = 7799, 4 right-hand sides from 739 to 425 us. The products in
// FP64 with the inverse in FP64 keep what substitution in FP32 gives and more: an inverse's error, eps64 cond(Op_qq),
// stays under eps32 up to condition 5e8, and measured against FP64 solves of the same factor the solution's error is
// 1.3e-7 against the substitution's 3.9e-7 on a board-like system of N = 3001, 6e-5 against 1e-4 on a random one (an
// inverse or W rounded to FP32 is not good enough: a factor whose pivots span 1e7 then preconditions poorly).
// The first blocks of a chain take the tile before theirs as any other one: W is ready 10 us after the inverse, and until
// then the longer step (2.4 us, without W) is the shorter way (N = 905: 109 us with W from the start, 89 so).
constexpr int FIRST = 6;
constexpr int S_LD = SB + 1;
constexpr size_t C64_LDS = 2 * SB * S_LD * sizeof(double2) + SB * sizeof(double2);

__device__ __forceinline__ void zfma(double &r, double &i, double2 a, double2 b)      // (r, i) += a b
{
    r = fma(a.x, b.x, fma(-a.y, b.y, r));
    i = fma(a.y, b.x, fma(a.x, b.y, i));
}

// X21 = -X22 (S21 X11) for the pairs of H x H blocks of S along the diagonal, X11 and X22 in place of theirs: NO rows of
// a column a thread, H / NO apart. S21 lies in S; the product S21 X11 goes there first.
template <int H> __device__ __forceinline__ void invert_level(double2 (*S)[S_LD], int tid)
{
    constexpr int NO = H == 32 ? 4 : H == 16 ? 2 : 1, NT = 32 * H / NO, ST = H / NO;
    const int p = tid / (NT / (SB / 2 / H)), x = tid % (NT / (SB / 2 / H)), i = x / H, j = x % H;
    double2(*M)[S_LD] = S + p * 2 * H;                       // the pair's corner
    const int c0 = p * 2 * H;
    double xr[NO], xi[NO];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        if (tid < NT) {
#pragma unroll
            for (int e = 0; e < NO; ++e) xr[e] = xi[e] = 0.0;
#pragma unroll 4
            for (int k = 0; k < H; ++k) {                    // triangular factors: zeros past the diagonal
                const double2 b = half ? M[H + k][c0 + j] : M[k][c0 + j];
#pragma unroll
                for (int e = 0; e < NO; ++e) zfma(xr[e], xi[e], M[H + i + ST * e][half ? c0 + H + k : c0 + k], b);
            }
        }
        __syncthreads();
        if (tid < NT) {
#pragma unroll
            for (int e = 0; e < NO; ++e)
                M[H + i + ST * e][c0 + j] = half ? make_double2(-xr[e], -xi[e]) : make_double2(xr[e], xi[e]);
        }
        __syncthreads();
    }
}

// The inverse of the lower triangular S (64 x 64, zeros above the diagonal) in place, rd holding the reciprocals of its
// diagonal: 8 x 8 blocks by substitution, a column a lane, then the blocks off the diagonal.
__device__ __forceinline__ void invert_lower(double2 (*S)[S_LD], const double2 *rd, int tid)
{
    if (tid < 64) {
        const int o = tid & ~7, j = tid & 7;
        double xr[8], xi[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            double sr = i == j ? 1.0 : 0.0, si = 0.0;
#pragma unroll
            for (int k = 0; k < i; ++k) {
                const double2 a = S[o + i][o + k];
                sr = fma(-a.x, xr[k], fma(a.y, xi[k], sr));
                si = fma(-a.y, xr[k], fma(-a.x, xi[k], si));
            }
            const double2 d = rd[o + i];
            xr[i] = sr * d.x - si * d.y;
            xi[i] = sr * d.y + si * d.x;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const bool in = i >= j;
            S[o + i][o + j] = make_double2(in ? xr[i] : 0.0, in ? xi[i] : 0.0);
        }
    }
    __syncthreads();
    invert_level<8>(S, tid);
    invert_level<16>(S, tid);
    invert_level<32>(S, tid);
}

// The products of the chain's steps. A wave has 16 rows of the operator, lane (cg, r) = (lane / 16, lane % 16) row r and
// columns 16 cg + v, and lane (cg, l) the vector's elements pair_col(h, lane) for right-hand side l % 2: the lanes of a
// column group then find its 16 pairs in their own DPP row, and a multiply-add takes them from there (row_newbcast) with
// no LDS read, exchange or barrier between a vector's arrival and the product. Written out because the compiler does not fold a 64-bit broadcast into the operation;
// the s_nop covers the two wait states between a vector write of x and its DPP read.
__device__ inline int pair_col(int h, int lane) { return (lane & 48) + 8 * h + ((lane & 15) >> 1); }
template <int N>
__device__ __forceinline__ void mac4(double (&a)[8], double xr, double xi, const double *wr, const double *wi)
{
    constexpr int n = 2 * (N & 7);
#define M25X_MAC(A0, A1, A2, A3, R, I, n0, n1, x, s)                                                         \
    "v_fmac_f64_dpp %" #A0 ", %" #x ", " s "%" #R " row_newbcast:%c" #n0 " row_mask:0xf bank_mask:0xf\n"     \
    "v_fmac_f64_dpp %" #A1 ", %" #x ", %" #I " row_newbcast:%c" #n0 " row_mask:0xf bank_mask:0xf\n"          \
    "v_fmac_f64_dpp %" #A2 ", %" #x ", " s "%" #R " row_newbcast:%c" #n1 " row_mask:0xf bank_mask:0xf\n"     \
    "v_fmac_f64_dpp %" #A3 ", %" #x ", %" #I " row_newbcast:%c" #n1 " row_mask:0xf bank_mask:0xf\n"
#define M25X_MAC2(R, I, n0, n1, R2, I2, m0, m1)                                                              \
    M25X_MAC(0, 1, 2, 3, R, I, n0, n1, 8, "") M25X_MAC(4, 5, 6, 7, R2, I2, m0, m1, 8, "")                    \
    M25X_MAC(0, 1, 2, 3, I, R, n0, n1, 9, "-") M25X_MAC(4, 5, 6, 7, I2, R2, m0, m1, 9, "-")
    asm("s_nop 1\n" M25X_MAC2(10, 14, 18, 19, 11, 15, 20, 21) M25X_MAC2(12, 16, 22, 23, 13, 17, 24, 25)
        : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7])
        : "v"(xr), "v"(xi), "v"(wr[N]), "v"(wr[N + 1]), "v"(wr[N + 2]), "v"(wr[N + 3]), "v"(wi[N]), "v"(wi[N + 1]),
          "v"(wi[N + 2]), "v"(wi[N + 3]), "n"(n), "n"(n + 1), "n"(n + 2), "n"(n + 3), "n"(n + 4), "n"(n + 5), "n"(n + 6),
          "n"(n + 7));
#undef M25X_MAC2
#undef M25X_MAC
}
// the sums over v and, by lane exchanges, over the four column groups: lane (cg, r) gets row r's real (cg even) or
// imaginary part for right-hand side cg / 2. Even and odd columns in sums of their own: eight chains of multiply-adds
// cover their latency.
__device__ __forceinline__ double rows_product(const float2 (&x)[2], const double *wr, const double *wi)
{
    const double r0 = (double)x[0].x, i0 = (double)x[0].y, r1 = (double)x[1].x, i1 = (double)x[1].y;
    double a[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    mac4<0>(a, r0, i0, wr, wi);
    mac4<4>(a, r0, i0, wr, wi);
    mac4<8>(a, r1, i1, wr, wi);
    mac4<12>(a, r1, i1, wr, wi);
#pragma unroll
    for (int e = 0; e < 4; ++e) a[e] += a[4 + e];
    return swap16_add(swap32_add(a[0], a[2]), swap32_add(a[1], a[3]));
}
// (wr, wi)[N + i] -= a x[N + i of the DPP row], i < 4: a row of W gains the multiple a of a row of the tile
template <int N> __device__ __forceinline__ void row_msub4(double *wr, double *wi, double2 x, double2 a)
{
#define M25X_MSUB(R, I, n)                                                                                   \
    "v_fmac_f64_dpp %" #R ", %8, -%10 row_newbcast:%c" #n " row_mask:0xf bank_mask:0xf\n"                    \
    "v_fmac_f64_dpp %" #I ", %8, -%11 row_newbcast:%c" #n " row_mask:0xf bank_mask:0xf\n"                    \
    "v_fmac_f64_dpp %" #R ", %9, %11 row_newbcast:%c" #n " row_mask:0xf bank_mask:0xf\n"                     \
    "v_fmac_f64_dpp %" #I ", %9, -%10 row_newbcast:%c" #n " row_mask:0xf bank_mask:0xf\n"
    asm("s_nop 1\n" M25X_MSUB(0, 4, 12) M25X_MSUB(1, 5, 13) M25X_MSUB(2, 6, 14) M25X_MSUB(3, 7, 15)
        : "+v"(wr[N]), "+v"(wr[N + 1]), "+v"(wr[N + 2]), "+v"(wr[N + 3]), "+v"(wi[N]), "+v"(wi[N + 1]), "+v"(wi[N + 2]),
          "+v"(wi[N + 3])
        : "v"(x.x), "v"(x.y), "v"(a.x), "v"(a.y), "n"(N), "n"(N + 1), "n"(N + 2), "n"(N + 3));
#undef M25X_MSUB
}
template <bool RM>
__device__ __forceinline__ void chain_of(const Tri<float2> &c, int q, Turn &turn)
{
    __shared__ __align__(16) unsigned char lds[C64_LDS];
    double2(*S)[S_LD] = (double2(*)[S_LD])lds;               // the triangle, then its inverse (solve order, lower)
    double2(*N)[S_LD] = S + SB;                              // the tile of the block before (rows in solve order)
    double2 *rd = (double2 *)(N + SB);
    const long n = c.n;
    const int nb = (int)((n + SB - 1) / SB);
    const bool fwd = c.fwd, unit = c.unit;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));            // (places worked out for each block: kept from block to block they are spilled)
    const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    auto order = [&](int p) { return fwd ? p : nb - 1 - p; };
    auto flip = [&](int i) { return fwd ? i : SB - 1 - i; };               // local row <-> its place in solve order
    const long r0 = (long)order(q) * SB;
    const int m = (int)std::min((long)SB, n - r0);                         // rows of this block inside the matrix
    const bool near = q > FIRST;
    const int nfar = near ? q - 1 : q;

    // the diagonal block and the tile before it, whole lines a load; indices clamped into the matrix
    float2 md[TE], mn[TE];
    const long kn = (long)order(near ? q - 1 : 0) * SB;
#pragma unroll
    for (int u = 0; u < TE; ++u) {
        const int i = RM ? wv * TE + u : lane, k = RM ? lane : wv * TE + u;
        const long gi = r0 + std::min(i, m - 1), gk = r0 + std::min(k, m - 1), gn = std::min(kn + k, n - 1);
        md[u] = RM ? c.LU[gi * c.lda + gk] : c.LU[gk * c.lda + gi];
        mn[u] = RM ? c.LU[gi * c.lda + gn] : c.LU[gn * c.lda + gi];
    }
    // waves 0-3 end with a row of -W each lane and finish the block, waves 4-7 with one of the inverse and form z
    const bool last = wv < 4;
    const int wi4 = wv & 3, li = 16 * wi4 + (lane & 15), gl = flip(li);    // the lane's row of the products
    const bool inrow = gl < m;
    const long grow = r0 + std::min(gl, m - 1);
    const long orow = last && c.out && c.operm ? c.operm[grow] : grow;
    constexpr int D = Depth<float2>::D;
    Tile<float2> t[D];
    far_begin<float2, RM>(t, c, nfar, r0, m, wv, lane, order);
#pragma unroll
    for (int u = 0; u < TE; ++u) {       // rows and columns past the matrix: those of the unit matrix
        const int i = RM ? wv * TE + u : lane, k = RM ? lane : wv * TE + u, si = flip(i), sk = flip(k);
        const bool in = i < m && k < m && (sk < si || (sk == si && !unit));
        double2 v = make_double2(in ? (double)md[u].x : 0.0, in ? (double)md[u].y : 0.0);
        if (si == sk) {
            if (!in) v.x = 1.0;
            rd[si] = trecip(v);
        }
        S[si][sk] = v;
        N[si][k] = make_double2(i < m ? (double)mn[u].x : 0.0, i < m ? (double)mn[u].y : 0.0);
    }
    __syncthreads();
    invert_lower(S, rd, tid);
    double wr[16], wi[16];                   // columns 16 (lane / 16) + v of row li
    const int cg16 = lane & 48;
    if (last) {
#pragma unroll
        for (int v = 0; v < 16; ++v) wr[v] = wi[v] = 0.0;
        if (near) {
#pragma unroll 2
            for (int k = 0; k < 16 * wi4 + 16; ++k) {        // the inverse is zero past its diagonal
                const double2 a = S[li][k], x = N[k][lane];
                row_msub4<0>(wr, wi, x, a);
                row_msub4<4>(wr, wi, x, a);
                row_msub4<8>(wr, wi, x, a);
                row_msub4<12>(wr, wi, x, a);
            }
        }
    } else {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const double2 a = S[li][cg16 + v];
            wr[v] = a.x;
            wi[v] = a.y;
        }
    }
    float2 bx[2];                            // waves 4-7: the right-hand sides of places pair_col(h, lane)
    const long b0 = r0 + std::min(flip(pair_col(0, lane)), m - 1), b1 = r0 + std::min(flip(pair_col(1, lane)), m - 1);
    if (!last && !c.wait) rhs_pair(c, b0, b1, lane & 1, bx);
    if (!turn.go()) return;
    if (!last && c.wait) rhs_pair(c, b0, b1, lane & 1, bx);
    __syncthreads();
    float4(*red)[SB] = (float4(*)[SB])lds;                                 // [wave][place]: partial sums of the pair
    u64(*zs)[64] = (u64(*)[64])(red + NWV);                                // z, as rows_product leaves it; set when written
    if (last) zs[wv][lane] = UNSET;
    {
        float o[2 * CR];
        const int i = far_sum<float2, RM>(o, t, c, q, nfar, r0, m, wv, lane, order);
        red[wv][flip(i)] = make_float4(o[0], o[1], o[2], o[3]);
    }
    __syncthreads();
    float2 y[2];
    if (!last) {                             // z = inv(Op_qq) (b - the far sum): the 8 waves' parts meet in every wave
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = pair_col(h, lane);
            float2 g[NWV];
#pragma unroll
            for (int w = 0; w < NWV; ++w) g[w] = ((const float2 *)&red[w][k])[lane & 1];
#pragma unroll
            for (int st = 1; st < NWV; st *= 2)
#pragma unroll
                for (int w = 0; w + st < NWV; w += 2 * st) g[w] = tadd(g[w], g[w + st]);
            y[h] = csel(flip(k) < m, tadd(bx[h], g[0]), make_float2(0.f, 0.f));
        }
        __builtin_amdgcn_s_setprio(2);
        const double z = rows_product(y, wr, wi);
        __hip_atomic_store(&zs[wi4][lane], mark_safe((u64)__double_as_longlong(z), 0x7ff8000000000000ull),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);       // lane's word of z, marked as y's are
        return;
    }
    __builtin_amdgcn_s_setprio(3);
    double x = 0.0;
    if (near) {                              // y = z - W y of the block before
        const long g0 = kn + pair_col(0, lane), g1 = kn + pair_col(1, lane);
        const float2 *p0 = c.dst + std::min(g0, n - 1) * CR + (lane & 1), *p1 = c.dst + std::min(g1, n - 1) * CR + (lane & 1);
        auto attempt = [&]() {
            const bool a0 = take(p0, y[0]), a1 = take(p1, y[1]);
            return a0 && a1;
        };
        wave_wait<true>(attempt(), c.abort, attempt);
        y[0] = csel(g0 < n, y[0], make_float2(0.f, 0.f));
        y[1] = csel(g1 < n, y[1], make_float2(0.f, 0.f));
        x = rows_product(y, wr, wi);
    }
    u64 z = UNSET;
    auto got_z = [&]() {
        z = __hip_atomic_load(&zs[wi4][lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        return z != UNSET;
    };
    wave_wait<false>(got_z(), c.abort, got_z);
    const unsigned f = __float_as_uint((float)(x + __longlong_as_double((long long)z)));
    const auto both = __builtin_amdgcn_permlane16_swap(f, f, false, false);    // even column groups: (re, im)
    if (inrow && !(lane & 16)) to_out(c, grow, orow, lane >> 5, make_float2(__uint_as_float(both[0]), __uint_as_float(both[1])));
}

// -- complex128 --
// The diagonal blocks by substitution (an inverse in the same precision as the factor would lose the accuracy of one
// with small pivots). Unit-lower (FWD) or unit-upper substitution of one right-hand side, lane i row i, with the
// block's operator Ms in LDS (rows pre-scaled to a unit diagonal; the diagonal, the other triangle and the padding
// zero): step k broadcasts y_k and every lane subtracts its multiple, the zeros leaving the finished rows alone. After
// each 8 steps the 8 rows they finished (lanes [lo, lo + 8)) are final: pub(lo) hands them on while the rest go on. The
// row's operator entries are read from LDS one group of 8 steps ahead.
template <bool FWD, class Pub>
__device__ __attribute__((always_inline)) void subst(double2 &t, const double2 (*Ms)[SB + 1], int lane, Pub &pub)
{
    double2 mk[2][8];
#pragma unroll
    for (int j = 0; j < 8; ++j) mk[0][j] = Ms[lane][FWD ? j : SB - 1 - j];
#pragma unroll
    for (int s0 = 0; s0 < SB; s0 += 8) {
        const int g = (s0 / 8) & 1;
        if (s0 + 8 < SB) {
#pragma unroll
            for (int j = 0; j < 8; ++j) mk[g ^ 1][j] = Ms[lane][FWD ? s0 + 8 + j : SB - 9 - s0 - j];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int k = FWD ? s0 + j : SB - 1 - s0 - j;
            t = tfms(t, mk[g][j], readlane_c(t, k));
        }
        pub(FWD ? s0 : SB - 8 - s0);
    }
}

// Workgroup q stages its diagonal block's operator in LDS (strict triangle, rows scaled by 1 / U_ii), sums the earlier
// blocks' part, and waves 0 and 1 form the block's right-hand sides (one each; lane i row i), substitute, and publish y_q
// eight rows at a time as the substitution finishes them: the next workgroup's wave that takes those rows starts its
// product with them while the substitution goes on, so the chain's hand-off overlaps the substitution.
// Two right-hand sides to a chain: a call of 5 to 8 ran as two calls of 4 one after the other, and the products of 4
// took 0.25 us more of a block's step than those of 2. N = 3001, 7 right-hand sides: 650 -> 333 us, 3.3 us
// a block, of which the substitution is 1.8.
template <bool RM>
__device__ __forceinline__ void chain_of(const Tri<double2> &c, int q, Turn &turn)
{
    typedef double2 T;
    __shared__ T Ms[SB][SB + 1];             // the diagonal block's operator
    __shared__ T red[NWV][CR][SB];           // the waves' partial sums
    // the right-hand sides and 1 / U_ii of the rows (past n: zeroed where used), parked in LDS until the substitution:
    // held in registers across the loop they are spilled to scratch, and reloading them would put a memory round trip
    // into every step of the chain
    __shared__ T bxs[CR][SB], rds[SB];
    const T *LU = c.LU;
    const long n = c.n, lda = c.lda;
    const int nb = (int)((n + SB - 1) / SB);
    const bool fwd = c.fwd, unit = c.unit;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));            // (places worked out for each block: kept from block to block they are spilled)
    const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const T zero = make_double2(0, 0), one = make_double2(1, 0);
    auto order = [&](int p) { return fwd ? p : nb - 1 - p; };
    auto opp = [&](long gi, long gk) { return RM ? LU + gi * lda + gk : LU + gk * lda + gi; };
    const long r0 = (long)order(q) * SB;
    const int m = (int)std::min((long)SB, n - r0);          // rows of this block inside the matrix

    // the diagonal block: thread (rows 8 wv + u, column lane) of a row-major operator, (row lane, columns 8 wv + u)
    // of a column-major one, so that every load reads whole lines; indices clamped into the block, the entries
    // outside it or outside the strict triangle zeroed when staged
    T md[TE];
#pragma unroll
    for (int u = 0; u < TE; ++u) {
        const int i = RM ? wv * TE + u : lane, k = RM ? lane : wv * TE + u;
        md[u] = *opp(r0 + std::min(i, m - 1), r0 + std::min(k, m - 1));
    }
    const long grow = r0 + std::min(lane, m - 1);
    if (wv == 0) rds[lane] = csel(unit, one, trecip(*opp(grow, grow)));
    constexpr int D = Depth<T>::D;
    Tile<T> t[D];
    far_begin<T, RM>(t, c, q, r0, m, wv, lane, order);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < TE; ++u) {
        const int i = RM ? wv * TE + u : lane, k = RM ? lane : wv * TE + u;
        const bool in = i < m && k < m && (fwd ? k < i : k > i);
        Ms[i][k] = csel(in, csel(unit, md[u], tmul(md[u], rds[i])), zero);
    }
    if (!turn.go()) return;
    if (wv == 0) {
        T b[CR];
        rhs_row(c, grow, b);
        bxs[0][lane] = b[0];
        bxs[1][lane] = b[1];
    }
    {
        double o[2 * CR];
        const int i = far_sum<T, RM>(o, t, c, q, q, r0, m, wv, lane, order);
        red[wv][0][i] = make_double2(o[0], o[1]);
        red[wv][1][i] = make_double2(o[2], o[3]);
    }
    __syncthreads();
    if (wv >= CR) return;
    const bool inrow = lane < m;
    T h[NWV];                                // the 8 waves' partial sums, added as a tree (depth 3)
#pragma unroll
    for (int sl = 0; sl < NWV; ++sl) h[sl] = red[sl][wv][lane];
#pragma unroll
    for (int st = 1; st < NWV; st *= 2)
#pragma unroll
        for (int sl = 0; sl + st < NWV; sl += 2 * st) h[sl] = tadd(h[sl], h[sl + st]);
    T y = csel(inrow, tmul(tadd(bxs[wv][lane], h[0]), rds[lane]), zero);
    auto pub = [&](int lo) __attribute__((always_inline)) {
        if (lane >= lo && lane < lo + 8 && inrow) put(c.dst + grow * CR + wv, y);
    };
    if (fwd) subst<true>(y, Ms, lane, pub);
    else subst<false>(y, Ms, lane, pub);
    if (inrow && c.out && wv < c.kc) c.out[(c.operm ? (long)c.operm[grow] : grow) * c.ldo + wv] = y;
}

template <typename T> struct Solve {     // a call's arguments and a workgroup's place in it
    const T *LU;
    long lda, n;
    T *B;
    long ldb;
    const int *perm;
    T *W1, *W2;
    int *abort;
    Held h;
    int nrhs, chain, own, pad;
};
// block i (both passes in order) of the chain: pass 0 reads B, pass 1 the solution of pass 0 and also writes B (every
// workgroup that reads a row of B has done so before the second pass has a solution for it: that needs the first pass's
// last block)
template <typename T> __device__ __forceinline__ Tri<T> chain_args(const Solve<T> &v, int pass, int trans)
{
    Tri<T> c;
    T *Bc = v.B + v.chain * CR;
    c.LU = v.LU; c.lda = v.lda; c.n = v.n;
    c.kc = std::min(CR, v.nrhs - v.chain * CR);
    c.fwd = pass == 0;                       // U^T, then L^T (row-major: RM); or L, then U
    c.unit = pass == trans;
    c.abort = v.abort;
    c.wait = pass;
    c.src = pass ? v.W1 + v.chain * CR * v.n : Bc;
    c.lds = v.ldb;
    c.sperm = pass || trans ? nullptr : v.perm;
    c.dst = (pass ? v.W2 : v.W1) + v.chain * CR * v.n;
    c.out = pass ? Bc : nullptr;
    c.ldo = v.ldb;
    c.operm = pass && trans ? v.perm : nullptr;
    return c;
}

// p, which came through LDS, known to the compiler to be in global memory (else its loads become flat ones)
template <typename P> __device__ __forceinline__ P *in_global(P *p)
{
    return (P *)(__attribute__((address_space(1))) P *)(u64)p;
}

// RM: the operator's rows are contiguous (trans = 1: U^T then L^T in the factor's row-major buffer). The workgroup's own
// block, where another one stays away that one's first. The arguments come back from LDS before a further block: held in
// scalar registers over a block they are spilled (20 of them, and a complex64 solve takes 2 to 4 % longer).
template <typename T, bool RM>
__device__ __forceinline__ void trsv_body(Solve<T> v, const ChainPos &at, u64 *held)
{
    __shared__ Solve<T> kept;
    const int nb = (int)((v.n + SB - 1) / SB);
    if (at.q >= nb) return;
    v.chain = at.chain;
    v.own = at.pass * nb + at.q;
    v.h = held_of(held, at.chain, nb);
    if (threadIdx.x == 0) {
        start_block(v.h, v.own);
        kept = v;
    }
    for (int i = v.own;;) {
        const int nbv = (int)((v.n + SB - 1) / SB), pass = i >= nbv;
        Turn turn{v.h, v.own, i, i};
        chain_of<RM>(chain_args(v, pass, (int)RM), i - pass * nbv, turn);
        if (turn.next < 0 || (turn.next == i && i == turn.own)) return;
        __builtin_amdgcn_s_setprio(0);
        __syncthreads();                     // every wave is done with the block's LDS
        constexpr int NW = sizeof(Solve<T>) / 4;
        int w[NW];
#pragma unroll
        for (int u = 0; u < NW; ++u) w[u] = __builtin_amdgcn_readfirstlane(((const int *)&kept)[u]);
        __builtin_memcpy(&v, w, sizeof v);
        v.LU = in_global(v.LU); v.B = in_global(v.B); v.perm = in_global(v.perm); v.W1 = in_global(v.W1);
        v.W2 = in_global(v.W2); v.abort = in_global(v.abort);
        v.h = Held{in_global(v.h.started), in_global(v.h.taken)};
        i = turn.next == i ? v.own : turn.next;
    }
}

template <typename T, bool RM>
__global__ __launch_bounds__(TB) void k_trsv(Solve<T> v, u64 *held)
{
    trsv_body<T, RM>(v, chain_pos(blockIdx.x, (int)((v.n + SB - 1) / SB), (v.nrhs + CR - 1) / CR), held);
}

// UNSET words to the first n words of each of gridDim.y buffers; the nheld words of the chains' blocks 0
__global__ void k_fill_unset(u64 *p, long pitch, long n, u64 *held, int nheld)
{
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < nheld && blockIdx.y == 0) held[i] = 0;
    if (i < n) p[blockIdx.y * pitch + i] = UNSET;
}

inline unsigned blocks(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

template <typename T> size_t work_bytes(long n)
{
    const int cus = 256;
    return 2 * (size_t)cus * sizeof(Slot<T>) + 2 * NB * sizeof(T) + 256;
}

template <typename T> int max_rows()
{
    // LDS for the slab: at most 128 KB
    return (int)((128 * 1024) / (NB * sizeof(T)));
}

template <typename T>
int getrf_t(T *A, long n, long lda, int *ipiv, int *info, void *work, size_t wbytes, hipStream_t s)
{
    if (wbytes < work_bytes<T>(n)) return fail(M25X_EINVAL, "getrf: workspace of %zu bytes, %zu needed", wbytes, work_bytes<T>(n));
    const int cus = std::min(num_cus(), 256);
    char *w = (char *)work;
    Slot<T> *slots = (Slot<T> *)w;
    T *diag = (T *)(w + 2 * (size_t)256 * sizeof(Slot<T>));
    Bar *bar = (Bar *)(w + 2 * (size_t)256 * sizeof(Slot<T>) + 2 * NB * sizeof(T));
    const int Rmax = max_rows<T>();
    static bool attr_done[2] = {false, false};
    const size_t smem_max = (size_t)Rmax * NB * sizeof(T);
    {
        static std::mutex mu;
        std::lock_guard<std::mutex> lk(mu);
        if (!attr_done[sizeof(T) == 8]) {
            M25X_HIP(hipFuncSetAttribute((const void *)k_panel<T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem_max));
            attr_done[sizeof(T) == 8] = true;
        }
    }
    if (info) {
        hipLaunchKernelGGL(k_zero_ints, dim3(1), dim3(64), 0, s, info, 1);
        if (int rc = check_launch("getrf")) return rc;
    }
    for (long j0 = 0; j0 < n; j0 += NB) {
        const int jb = (int)std::min((long)NB, n - j0);
        const long m = n - j0;
        int G = (int)std::min((long)cus, (m + Rmax - 1) / Rmax);
        G = std::max(G, 1);
        int R = (int)((m + G - 1) / G);
        hipLaunchKernelGGL(k_zero_ints, dim3(1), dim3(64), 0, s, (int *)bar, 4);
        if (int rc = check_launch("getrf")) return rc;
        const size_t smem = (size_t)R * jb * sizeof(T);
        void *args[] = {(void *)&A, (void *)&lda, (void *)&n, (void *)&j0, (void *)&jb, (void *)&R, (void *)&ipiv,
                        (void *)&info, (void *)&slots, (void *)&diag, (void *)&bar};
        const int dt = dtype_of<T>();
        const double es = sizeof(T);
        {
            TimedLaunch tl(s, M25X_K_PANEL, dt, 2.0 * es * m * jb, 0.0);
            M25X_HIP(hipLaunchCooperativeKernel((const void *)k_panel<T>, dim3(G), dim3(PT), args, (unsigned)smem, s));
        }
        const long nsw = n - jb;
        if (nsw > 0) {
            TimedLaunch tl(s, M25X_K_LASWP, dt, 2.0 * es * 2 * jb * nsw, 0.0);
            hipLaunchKernelGGL(k_laswp<T>, dim3(blocks(nsw, 256)), dim3(256), 0, s, A, lda, n, j0, jb, ipiv);
            if (int rc = check_launch("getrf/laswp")) return rc;
        }
        const long c0 = j0 + jb;
        if (c0 < n) {
            {
                TimedLaunch tl(s, M25X_K_TRSM, dt, 2.0 * es * (n - c0) * jb, 4.0 * (n - c0) * jb * jb);
                hipLaunchKernelGGL(k_trsm<T>, dim3(blocks(n - c0, TC)), dim3(256), 0, s, A, lda, n, j0, jb, c0);
            }
            if (int rc = check_launch("getrf/trsm")) return rc;
            const long M = n - c0;
            {
                TimedLaunch tl(s, M25X_K_GEMM, dt, es * (2.0 * M * M + 2.0 * M * jb), 8.0 * M * M * jb);
                hipLaunchKernelGGL((k_gemm<T>), dim3(gemm_grid(M, M)), dim3(GT), 0, s, A + c0 * lda + c0, lda, A + j0 * lda + c0,
                                   lda, A + c0 * lda + j0, lda, M, M, (long)jb);
            }
            if (int rc = check_launch("getrf/gemm")) return rc;
        }
    }
    return M25X_OK;
}

// ---- look-ahead: the next panel's tournament beside the trailing update -----------------------------------
// The tournament of panel j + 1 needs only panel j + 1's columns updated, so the update of step j is split: the next
// panel's 64 columns first, on the caller's stream, with the tournament right behind them, and the rest on a side stream
// that waits for those columns. A tournament workgroup takes all registers of a CU, so it can start only on an empty
// one: in this order its workgroups are there before the rest of the update is let go. (The other way round, the
// tournament on the side stream, it waits for the update's thousands of workgroups to drain and nothing is gained.)
// N = 7799: complex64 43.3 -> 36.5 ms, complex128 58.7 -> 49.3; N = 14 000, complex64: 139 -> 120 ms. Beside the update
// a tournament takes 1.5 to 1.7 times as long (the clock falls to 2.2 GHz, 1.95 for complex128, and its 53 KB of code
// share an instruction cache with the update on the CU next to it) and the update 1.2 times.
// On by default (m25x_lu_set_lookahead).
std::atomic<int> g_lookahead{1};

// A side stream and its events, leased to one call at a time (what a call has enqueued keeps its order on the stream
// when the next lease goes on). At most MAX_SIDE a device, made as calls need them and kept.
struct Side {
    hipStream_t s = nullptr;
    hipEvent_t next = nullptr, done = nullptr;
};
constexpr int MAX_SIDE = 4, SIDE_DEVICES = 64;
struct SidePool {
    std::mutex mu;
    Side side[MAX_SIDE];
    int made = 0;
    unsigned busy = 0;
};
SidePool side_pool[SIDE_DEVICES];

class SideLease {
public:
    // For work on `caller`; empty (use one stream) if not wanted, look-ahead is off, the caller's stream is being captured (a leased
    // stream would stay part of the capture after the call), or none is free or can be made.
    SideLease(hipStream_t caller, bool wanted)
    {
        int dev = -1;
        hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
        if (!wanted || !g_lookahead.load(std::memory_order_relaxed)) return;
        if (hipStreamIsCapturing(caller, &st) != hipSuccess || st != hipStreamCaptureStatusNone ||
            hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= SIDE_DEVICES) {
            (void)hipGetLastError();
            return;
        }
        SidePool &p = side_pool[dev];
        std::lock_guard<std::mutex> lk(p.mu);
        for (int i = 0; i < MAX_SIDE; ++i) {
            if (p.busy >> i & 1) continue;
            if (i >= p.made) {
                Side n;
                if (hipStreamCreateWithFlags(&n.s, hipStreamNonBlocking) != hipSuccess ||
                    hipEventCreateWithFlags(&n.next, hipEventDisableTiming) != hipSuccess ||
                    hipEventCreateWithFlags(&n.done, hipEventDisableTiming) != hipSuccess) {
                    (void)hipGetLastError();
                    if (n.next) (void)hipEventDestroy(n.next);
                    if (n.s) (void)hipStreamDestroy(n.s);
                    return;
                }
                p.side[i] = n;
                p.made = i + 1;
            }
            p.busy |= 1u << i;
            pool = &p;
            index = i;
            return;
        }
    }
    ~SideLease()
    {
        if (!pool) return;
        std::lock_guard<std::mutex> lk(pool->mu);
        pool->busy &= ~(1u << index);
    }
    SideLease(const SideLease &) = delete;
    SideLease &operator=(const SideLease &) = delete;
    const Side *get() const { return pool ? &pool->side[index] : nullptr; }

private:
    SidePool *pool = nullptr;
    int index = 0;
};

// What a call has on its side stream: the caller's stream waits for it before the matrix is read again, and where the call
// ends early (a launch that fails), so that the matrix' memory is free to its owner in the caller's stream's order.
struct Beside {
    hipStream_t s;
    const Side *side;
    bool open = false;
    int join()
    {
        if (open && hipStreamWaitEvent(s, side->done, 0) != hipSuccess) return fail(M25X_EHIP, "getrf: wait");
        open = false;
        return M25X_OK;
    }
    ~Beside()
    {
        if (open && (hipEventRecord(side->done, side->s) != hipSuccess || hipStreamWaitEvent(s, side->done, 0) != hipSuccess))
            (void)hipStreamSynchronize(side->s);
    }
};

// From this many trailing rows on a step's update is split: below it the update is hardly longer than what the split
// costs (the extra launch and two events, about 25 us; at 2500 rows 7.48 ms without and 7.38 with it).
constexpr long LOOK_ROWS = 2048;

template <typename T> size_t tour_work_bytes(long n)
{
    const long nn = tour_nodes(n, Tour<T>::RL, Tour<T>::AR);
    return nn * sizeof(TNode<T>) + (size_t)TW * TW * sizeof(T) + sizeof(int) * ((size_t)nn + 4 * TW + 64);
}

// L21 and U12 of a panel of TW columns, m rows and columns beyond it: one launch
template <typename T> void launch_tri(hipStream_t s, T *A, long lda, long j0, long m, const T *top)
{
    TimedLaunch tl(s, M25X_K_L21, dtype_of<T>(), 4.0 * sizeof(T) * m * TW, 8.0 * m * TW * TW);
    hipLaunchKernelGGL(k_tri<T>, dim3(2 * blocks(m, TRI_N)), dim3(256), 0, s, A, lda, j0, m, top);
}

template <typename T>
int getrf_tp(T *A, long n, long lda, int *ipiv, int *perm, int *info, void *work, size_t wbytes, hipStream_t s)
{
    constexpr int RL = Tour<T>::RL, AR = Tour<T>::AR;
    if (wbytes < tour_work_bytes<T>(n))
        return fail(M25X_EINVAL, "getrf: workspace of %zu bytes, %zu needed", wbytes, tour_work_bytes<T>(n));
    const long nn = tour_nodes(n, RL, AR);
    char *w = (char *)work;
    TNode<T> *nodes = (TNode<T> *)w;
    w += nn * sizeof(TNode<T>);
    T *top = (T *)w;
    w += (size_t)TW * TW * sizeof(T);
    int *arrive = (int *)w, *pairs = arrive + nn;
    hipLaunchKernelGGL(k_zero_ints, dim3(blocks(nn, 256)), dim3(256), 0, s, arrive, (int)nn);
    if (info) hipLaunchKernelGGL(k_zero_ints, dim3(1), dim3(64), 0, s, info, 1);
    if (perm) hipLaunchKernelGGL(k_iota, dim3(blocks(n, 256)), dim3(256), 0, s, perm, n);
    if (int rc = check_launch("getrf")) return rc;
    const SideLease lease(s, n - TW >= LOOK_ROWS);
    const Side *side = lease.get();
    const int dt = dtype_of<T>();
    const double es = sizeof(T);
    auto tournament = [&](long j0) -> int {
        const int jb = (int)std::min((long)TW, n - j0);
        const long m = n - j0;
        TimedLaunch tl(s, M25X_K_TSLU, dt, es * m * jb, 0.0);
        return launch_tslu((const T *)A, lda, n, j0, jb, (int)tour_leaves(m, RL), nodes, arrive, top, ipiv, pairs, info, s);
    };
    auto update = [&](hipStream_t on, long j0, int jb, long c1, long c2) {      // A22[:, c1:c2] -= L21 U12[:, c1:c2]
        const long c0 = j0 + jb, M = n - c0, N = c2 - c1;
        TimedLaunch tl(on, M25X_K_GEMM, dt, es * (2.0 * M * N + (double)(M + N) * jb), 8.0 * M * N * jb);
        launch_update<T>(on, A + c1 * lda + c0, lda, (const T *)(A + j0 * lda + c0), lda, (const T *)(A + c1 * lda + j0),
                         lda, M, N, (long)jb);
    };
    if (int rc = tournament(0)) return rc;
    Beside beside{s, side};                  // the last update's rest, where it runs on the side stream
    for (long j0 = 0; j0 < n; j0 += TW) {
        const int jb = (int)std::min((long)TW, n - j0);
        if (int rc = beside.join()) return rc;
        {
            TimedLaunch tl(s, M25X_K_APPLY_MOVES, dt, 2.0 * es * 2 * jb * n, 0.0);
            hipLaunchKernelGGL(k_apply_moves<T>, dim3(blocks(n, 8) + (perm ? 1 : 0)), dim3(256), 0, s, A, lda, 0L, n,
                               (const int *)pairs, j0, jb, (const T *)top, perm);
        }
        if (int rc = check_launch("getrf/panel")) return rc;
        const long c0 = j0 + jb;
        if (c0 >= n) break;
        launch_tri(s, A, lda, j0, n - c0, (const T *)top);   // L21 = A21 U11^-1 and U12 = L11^-1 A12
        if (side && n - c0 >= LOOK_ROWS) {
            const long c1 = c0 + TW;
            update(s, j0, jb, c0, c1);                       // the next panel's columns
            if (hipEventRecord(side->next, s) != hipSuccess || hipStreamWaitEvent(side->s, side->next, 0) != hipSuccess)
                return fail(M25X_EHIP, "getrf: look-ahead");
            if (int rc = tournament(c0)) return rc;          // in place before the rest is let go
            beside.open = true;
            update(side->s, j0, jb, c1, n);
            if (hipEventRecord(side->done, side->s) != hipSuccess) return fail(M25X_EHIP, "getrf: look-ahead");
        } else {
            update(s, j0, jb, c0, n);
            if (int rc = tournament(c0)) return rc;
        }
        if (int rc = check_launch("getrf/update")) return rc;
    }
    return M25X_OK;
}

// Solve workspace: y of the two solves (W1, W2: n x MAXRHS each), written as self-marking values over UNSET words; the
// words of the chains' blocks, in room for a third such buffer and n values (with that room the size is what it has been:
// the largest n that m25x_getrs_noalloc takes follows from it); the permutation, the abort word (at the passed
// work_bytes - 256, rounded down to an int: callers read it there) and 63 spare ints.
template <typename T> size_t getrs_work(long n, long)
{
    return sizeof(T) * (3 * (size_t)n * MAXRHS + (size_t)n) + sizeof(int) * ((size_t)n + 64);
}
template <typename T> struct RsWork {
    T *W1, *W2;
    u64 *held;
    int *perm;
};
template <typename T> __host__ __device__ inline RsWork<T> rs_carve(void *work, long n)
{
    const size_t wn = (size_t)n * MAXRHS;
    T *w = (T *)work;
    return RsWork<T>{w, w + wn, (u64 *)(w + 2 * wn), (int *)(w + 3 * wn + n)};
}

// The solve with the buffers at buf (getrs_work(n) - 256 bytes) and the abort word given (not reset here).
template <typename T>
int getrs_noreset(const T *LU, long n, long lda, const int *ipiv, const int *perm, T *B, long ldb, int nrhs, int trans,
                  char *buf, int *abort, hipStream_t s)
{
    trans = trans != 0;
    const RsWork<T> w = rs_carve<T>(buf, n);
    const int nb = (int)((n + SB - 1) / SB), nchain = (nrhs + CR - 1) / CR;
    if (!perm) {
        hipLaunchKernelGGL(k_perm, dim3(1), dim3(256), 0, s, ipiv, n, w.perm);
        perm = w.perm;
    }
    const long words = (long)(nchain * CR * sizeof(T) / 8) * n;
    hipLaunchKernelGGL(k_fill_unset, dim3(blocks(words, 256), 2), dim3(256), 0, s, (u64 *)w.W1,
                       (long)((w.W2 - w.W1) * sizeof(T) / 8), words, w.held, 2 * nchain * held_words(nb));
    if (int rc = check_launch("getrs")) return rc;
    TimedLaunch tl(s, M25X_K_TRSV, dtype_of<T>(), ((double)n * n + 4.0 * n * nrhs) * sizeof(T), 8.0 * n * n * nrhs);
    const dim3 grid(2 * chain_wgs(nb, nchain));
    const Solve<T> v{LU, lda, n, B, ldb, perm, w.W1, w.W2, abort, {}, nrhs};
    if (trans) hipLaunchKernelGGL((k_trsv<T, true>), grid, dim3(TB), 0, s, v, w.held);
    else hipLaunchKernelGGL((k_trsv<T, false>), grid, dim3(TB), 0, s, v, w.held);
    return check_launch("getrs/trsv");
}

// The solve: buffers carved from `work`, the abort word at work + wbytes - 256 (rounded down to an int), zeroed once
// here and raised by any chain whose wait ran out.
template <typename T>
int getrs_t(const T *LU, long n, long lda, const int *ipiv, const int *perm_in, T *B, long ldb, int nrhs, int trans,
            void *work, size_t wbytes, hipStream_t s)
{
    if (nrhs < 1 || nrhs > MAXRHS) return fail(M25X_EINVAL, "getrs: 1 to %d right-hand sides, not %d", MAXRHS, nrhs);
    if (ldb < nrhs) return fail(M25X_EINVAL, "getrs: ldb < nrhs");
    if (!work || wbytes < getrs_work<T>(n, ldb))
        return fail(M25X_EINVAL, "getrs: workspace of %zu bytes, %zu needed", wbytes, getrs_work<T>(n, ldb));
    int *abort = (int *)((char *)work + ((wbytes - 256) & ~(size_t)3));
    hipLaunchKernelGGL(k_zero_ints, dim3(1), dim3(64), 0, s, abort, 1);
    return getrs_noreset<T>(LU, n, lda, ipiv, perm_in, B, ldb, nrhs, trans, (char *)work, abort, s);
}

// ---- batches ------------------------------------------------------------------------------------------------
// Every kernel of a panel step (or of a solve) once for all items of a batch: grid rows (or the last grid
// dimension) over the items, each workgroup reading its item from the item table; workgroups past an item's own
// extent, and items already done, leave at once. The items' results are those of the one-matrix calls.

// the tournament counters zeroed, info cleared, perm = 0 .. n - 1
template <typename T>
__global__ void k_lu_init_b(const m25x_lu_item *items)
{
    const m25x_lu_item it = items[blockIdx.y];
    const TourWork<T> w = tour_carve<T>(it.work, it.n);
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < w.nn) w.arrive[i] = 0;
    if (it.perm && i < it.n) it.perm[i] = (int)i;
    if (i == 0 && it.info) *it.info = 0;
}

template <typename T>
__global__ __launch_bounds__(256) void k_apply_moves_b(const m25x_lu_item *items, long j0)
{
    const m25x_lu_item it = items[blockIdx.y];
    const long n = it.n;
    if (j0 >= n) return;
    const long nb = (n + 7) / 8;
    if ((long)blockIdx.x > nb || ((long)blockIdx.x == nb && !it.perm)) return;
    const TourWork<T> w = tour_carve<T>(it.work, n);
    apply_moves_body<T>((T *)it.A, it.lda, 0, n, w.pairs, j0, (int)std::min((long)TW, n - j0), w.top, it.perm,
                        blockIdx.x, nb);
}

template <typename T>
__global__ __launch_bounds__(256) void k_tri_b(const m25x_lu_item *items, long j0)
{
    const m25x_lu_item it = items[blockIdx.y];
    const long m = it.n - j0 - TW, nb21 = (m + TRI_N - 1) / TRI_N;
    if (m <= 0 || (long)blockIdx.x >= 2 * nb21) return;
    const TourWork<T> w = tour_carve<T>(it.work, it.n);
    tri_body<T>((T *)it.A, it.lda, j0, m, (const T *)w.top, blockIdx.x, nb21);
}

template <typename T, int KS, typename AC = double2>
__global__ __launch_bounds__(GT) void k_gemm_b(const m25x_lu_item *items, long j0)
{
    const m25x_lu_item it = items[blockIdx.z];
    const long n = it.n;
    if (j0 >= n) return;
    const int jb = (int)std::min((long)TW, n - j0);
    const long c0 = j0 + jb, M = n - c0;
    if (M <= 0 || (long)blockIdx.x * GM >= M || (long)blockIdx.y * GN >= M) return;
    T *A = (T *)it.A;
    const long lda = it.lda;
    gemm_body<T, AC, KS>(A + c0 * lda + c0, lda, A + j0 * lda + c0, lda, A + c0 * lda + j0, lda, M, M, jb,
                               blockIdx.x, blockIdx.y);
}

template <typename T>
int getrf_batched_t(int nitems, const m25x_lu_item *h, const m25x_lu_item *d, hipStream_t s)
{
    long nmax = 0, work_max = 1;
    bool sorted = true;
    for (int i = 0; i < nitems; ++i) {
        const m25x_lu_item &it = h[i];
        if (!it.A || !it.ipiv || !it.work || it.n < 0 || it.lda < it.n || it.n > (1L << 30))
            return fail(M25X_EINVAL, "getrf_batched: item %d: bad arguments", i);
        if (it.work_bytes < tour_work_bytes<T>(it.n))
            return fail(M25X_EINVAL, "getrf_batched: item %d: workspace of %zu bytes, %zu needed", i, it.work_bytes,
                        tour_work_bytes<T>(it.n));
        nmax = std::max(nmax, it.n);
        work_max = std::max(work_max, std::max(it.n, tour_nodes(it.n, Tour<T>::RL, Tour<T>::AR)));
        if (i && it.n > h[i - 1].n) sorted = false;
    }
    if (nitems == 0 || nmax == 0) return M25X_OK;
    const int dt = dtype_of<T>();
    const double es = sizeof(T);
    hipLaunchKernelGGL(k_lu_init_b<T>, dim3(blocks(work_max, 256), nitems), dim3(256), 0, s, d);
    if (int rc = check_launch("getrf_batched")) return rc;
    int na = nitems;
    for (long j0 = 0; j0 < nmax; j0 += TW) {
        // the items still in the factorisation: a prefix when sorted by size (the grids then shrink with them)
        while (sorted && na > 0 && h[na - 1].n <= j0) --na;
        const long nbig = sorted ? h[0].n : nmax, mbig = nbig - j0;
        double flops = 0, pbytes = 0;
        for (int i = 0; i < na; ++i) {
            const long n = h[i].n;
            if (j0 >= n) continue;
            const long jb = std::min((long)TW, n - j0), M = n - j0 - jb;
            flops += 8.0 * M * M * jb;
            pbytes += es * (n - j0) * jb;
        }
        {
            TimedLaunch tl(s, M25X_K_TSLU, dt, pbytes, 0.0);
            if (int rc = launch_tslu_b((const T *)nullptr, d, na, j0, (int)tour_leaves(mbig, Tour<T>::RL), s))
                return rc;
        }
        hipLaunchKernelGGL(k_apply_moves_b<T>, dim3(blocks(nbig, 8) + 1, na), dim3(256), 0, s, d, j0);
        if (int rc = check_launch("getrf_batched/panel")) return rc;
        if (mbig > TW) {
            hipLaunchKernelGGL(k_tri_b<T>, dim3(2 * blocks(mbig - TW, TRI_N), na), dim3(256), 0, s, d, j0);
            TimedLaunch tl(s, M25X_K_GEMM, dt, 0.0, flops);
            const dim3 grid(blocks(mbig - TW, GM), blocks(mbig - TW, GN), na);
            const bool f32 = sizeof(T) == 8 && g_update_fp32.load(std::memory_order_relaxed);
            switch (g_gemm_stage.load(std::memory_order_relaxed)) {
            case 16:
                if (f32) hipLaunchKernelGGL((k_gemm_b<T, 16, float2>), grid, dim3(GT), 0, s, d, j0);
                else hipLaunchKernelGGL((k_gemm_b<T, 16>), grid, dim3(GT), 0, s, d, j0);
                break;
            case 32:
                if (f32) hipLaunchKernelGGL((k_gemm_b<T, 32, float2>), grid, dim3(GT), 0, s, d, j0);
                else hipLaunchKernelGGL((k_gemm_b<T, 32>), grid, dim3(GT), 0, s, d, j0);
                break;
            default:
                if (f32) hipLaunchKernelGGL((k_gemm_b<T, 8, float2>), grid, dim3(GT), 0, s, d, j0);
                else hipLaunchKernelGGL((k_gemm_b<T, 8>), grid, dim3(GT), 0, s, d, j0);
            }
        }
        if (int rc = check_launch("getrf_batched/update")) return rc;
    }
    return M25X_OK;
}

// W1, W2 of every item filled with UNSET words, the words of its chains' blocks 0
template <typename T>
__global__ void k_rs_prep_b(const m25x_rs_item *items)
{
    const m25x_rs_item it = items[blockIdx.y];
    const RsWork<T> w = rs_carve<T>(it.work, it.n);
    const long words = (long)((it.nrhs + CR - 1) / CR * CR * sizeof(T) / 8) * it.n;
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < words) ((u64 *)w.W1)[i] = ((u64 *)w.W2)[i] = UNSET;
    if (i < 2 * ((it.nrhs + CR - 1) / CR) * held_words((int)((it.n + SB - 1) / SB))) w.held[i] = 0;
}

// Both triangles of every item: workgroup g is workgroup g / nitems of item g % nitems (the chains side by side). nb,
// nchain: the most blocks and chains of an item.
template <typename T, bool RM>
__global__ __launch_bounds__(TB) void k_trsv_b(const m25x_rs_item *items, int nitems, int nb, int nchain, int *abort)
{
    const m25x_rs_item it = items[blockIdx.x % nitems];
    const ChainPos at = chain_pos(blockIdx.x / nitems, nb, nchain);
    if (at.chain * CR >= it.nrhs) return;
    const RsWork<T> w = rs_carve<T>(it.work, it.n);
    trsv_body<T, RM>(Solve<T>{(const T *)it.LU, it.lda, it.n, (T *)it.B, it.ldb, it.perm, w.W1, w.W2, abort, {}, it.nrhs},
                     at, w.held);
}

template <typename T>
int getrs_batched_t(int nitems, const m25x_rs_item *h, const m25x_rs_item *d, int trans, int *status, hipStream_t s)
{
    trans = trans != 0;
    long nmax = 0;
    int rmax = 0, nbmax = 0;
    for (int i = 0; i < nitems; ++i) {
        const m25x_rs_item &it = h[i];
        if (!it.LU || !it.perm || !it.B || !it.work || it.n < 0 || it.lda < it.n || it.nrhs < 1 ||
            it.nrhs > MAXRHS || it.ldb < it.nrhs)
            return fail(M25X_EINVAL, "getrs_batched: item %d: bad arguments (perm required, 1 <= nrhs <= %d)", i,
                        MAXRHS);
        if (it.work_bytes < getrs_work<T>(it.n, it.ldb))
            return fail(M25X_EINVAL, "getrs_batched: item %d: workspace of %zu bytes, %zu needed", i, it.work_bytes,
                        getrs_work<T>(it.n, it.ldb));
        nmax = std::max(nmax, it.n);
        rmax = std::max(rmax, it.nrhs);
        nbmax = std::max(nbmax, (int)((it.n + SB - 1) / SB));
    }
    hipLaunchKernelGGL(k_zero_ints, dim3(1), dim3(64), 0, s, status, 1);
    if (int rc = check_launch("getrs_batched")) return rc;
    if (nitems == 0 || nmax == 0) return M25X_OK;
    const int nchain = (rmax + CR - 1) / CR, dt = dtype_of<T>();
    hipLaunchKernelGGL(k_rs_prep_b<T>, dim3(blocks((long)(nchain * CR * sizeof(T) / 8) * nmax, 256), nitems), dim3(256), 0,
                       s, d);
    if (int rc = check_launch("getrs_batched")) return rc;
    double bytes = 0, flops = 0;
    for (int i = 0; i < nitems; ++i) {
        bytes += ((double)h[i].n * h[i].n + 4.0 * h[i].n * h[i].nrhs) * sizeof(T);
        flops += 8.0 * h[i].n * h[i].n * h[i].nrhs;
    }
    TimedLaunch tl(s, M25X_K_TRSV, dt, bytes, flops);
    const dim3 grid(2 * chain_wgs(nbmax, nchain) * nitems);
    if (trans) hipLaunchKernelGGL((k_trsv_b<T, true>), grid, dim3(TB), 0, s, d, nitems, nbmax, nchain, status);
    else hipLaunchKernelGGL((k_trsv_b<T, false>), grid, dim3(TB), 0, s, d, nitems, nbmax, nchain, status);
    return check_launch("getrs_batched/trsv");
}

// ---- the solve without allocation ------------------------------------------------------------------------
// The workspace of m25x_getrs_noalloc: one array per device, in the code object of this file, held until the process
// ends. Host code never passes the array's name to a kernel or a copy (on the host it is only a stand-in): the
// device address comes from hipGetSymbolAddress, once per device, and is kept in scratch_dev.
static __device__ __align__(256) unsigned char scratch[M25X_GETRS_SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
std::mutex scratch_mu;
void *scratch_dev[MAX_DEVICES];

// The current device's address of `scratch` (looked up at the first call on that device).
int scratch_of_current(char **out)
{
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES)
        return fail(M25X_EHIP, "getrs_noalloc: no current device");
    std::lock_guard<std::mutex> g(scratch_mu);
    if (!scratch_dev[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(M25X_EHIP, "getrs_noalloc: hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
        scratch_dev[dev] = p;
    }
    *out = (char *)scratch_dev[dev];
    return M25X_OK;
}

template <typename T>
int getrs_noalloc_t(const T *LU, long n, long lda, const int *ipiv, const int *perm_in, T *B, long ldb, int nrhs,
                    int trans, int *status, hipStream_t s)
{
    if (nrhs < 1 || nrhs > MAXRHS) return fail(M25X_EINVAL, "getrs_noalloc: 1 to %d right-hand sides, not %d", MAXRHS, nrhs);
    if (ldb < nrhs) return fail(M25X_EINVAL, "getrs_noalloc: ldb < nrhs");
    // the buffers getrs_noreset carves: getrs_work less its 256-byte tail
    const size_t need = getrs_work<T>(n, ldb) - 256;
    if (need > (size_t)M25X_GETRS_SCRATCH_BYTES)
        return fail(M25X_EINVAL, "getrs_noalloc: n = %ld needs %zu bytes of workspace, more than the %u held per device",
                    n, need, (unsigned)M25X_GETRS_SCRATCH_BYTES);
    char *buf = nullptr;
    if (int rc = scratch_of_current(&buf)) return rc;
    hipLaunchKernelGGL(k_zero_ints, dim3(1), dim3(64), 0, s, status, 1);
    if (int rc = check_launch("getrs_noalloc")) return rc;
    return getrs_noreset<T>(LU, n, lda, ipiv, perm_in, B, ldb, nrhs, trans, buf, status, s);
}

}  // namespace

extern "C" {

int m25x_lu_set_gemm_stage(int ks)
{
    if (ks != 8 && ks != 16 && ks != 32) return fail(M25X_EINVAL, "lu_set_gemm_stage: 8, 16 or 32, not %d", ks);
    g_gemm_stage.store(ks, std::memory_order_relaxed);
    return M25X_OK;
}

int m25x_lu_gemm_stage(void) { return g_gemm_stage.load(std::memory_order_relaxed); }

int m25x_lu_set_update_precision(int fp32)
{
    if (fp32 != 0 && fp32 != 1) return fail(M25X_EINVAL, "lu_set_update_precision: 0 (FP64) or 1 (FP32), not %d", fp32);
    g_update_fp32.store(fp32, std::memory_order_relaxed);
    return M25X_OK;
}

int m25x_getrf_batched(int dtype, int nitems, const m25x_lu_item *items_host, const m25x_lu_item *items_dev,
                       void *stream)
{
    if (nitems < 0 || (nitems && (!items_host || !items_dev))) return fail(M25X_EINVAL, "getrf_batched: bad arguments");
    hipStream_t s = (hipStream_t)stream;
    if (dtype == M25X_C128) return getrf_batched_t<double2>(nitems, items_host, items_dev, s);
    if (dtype == M25X_C64) return getrf_batched_t<float2>(nitems, items_host, items_dev, s);
    return fail(M25X_EINVAL, "getrf_batched: dtype %d", dtype);
}

int m25x_getrs_batched(int dtype, int nitems, const m25x_rs_item *items_host, const m25x_rs_item *items_dev, int trans,
                       int *status, void *stream)
{
    if (nitems < 0 || !status || (nitems && (!items_host || !items_dev)))
        return fail(M25X_EINVAL, "getrs_batched: bad arguments");
    hipStream_t s = (hipStream_t)stream;
    if (dtype == M25X_C128) return getrs_batched_t<double2>(nitems, items_host, items_dev, trans, status, s);
    if (dtype == M25X_C64) return getrs_batched_t<float2>(nitems, items_host, items_dev, trans, status, s);
    return fail(M25X_EINVAL, "getrs_batched: dtype %d", dtype);
}

int m25x_getrs_noalloc(int dtype, const void *LU, long n, long lda, const int *ipiv, const int *perm, void *B,
                       long ldb, int nrhs, int trans, int *status, void *stream)
{
    if (!LU || !ipiv || !B || !status || n < 0 || lda < n) return fail(M25X_EINVAL, "getrs_noalloc: bad arguments");
    if (dtype != M25X_C128 && dtype != M25X_C64) return fail(M25X_EINVAL, "getrs_noalloc: dtype %d", dtype);
    hipStream_t s = (hipStream_t)stream;
    if (n == 0) {
        hipLaunchKernelGGL(k_zero_ints, dim3(1), dim3(64), 0, s, status, 1);
        return check_launch("getrs_noalloc");
    }
    if (dtype == M25X_C128)
        return getrs_noalloc_t<double2>((const double2 *)LU, n, lda, ipiv, perm, (double2 *)B, ldb, nrhs, trans,
                                        status, s);
    return getrs_noalloc_t<float2>((const float2 *)LU, n, lda, ipiv, perm, (float2 *)B, ldb, nrhs, trans, status, s);
}

size_t m25x_getrf_work_bytes(int dtype, long n)
{
    return dtype == M25X_C64 ? std::max(work_bytes<float2>(n), tour_work_bytes<float2>(n))
                             : std::max(work_bytes<double2>(n), tour_work_bytes<double2>(n));
}

int m25x_getrf(int dtype, int pivot, void *A, long n, long lda, int *ipiv, int *perm, int *info, void *work,
               size_t wbytes, void *stream)
{
    if (!A || !ipiv || !work || n < 0 || lda < n) return fail(M25X_EINVAL, "getrf: bad arguments");
    if (pivot != M25X_PIVOT_PARTIAL && pivot != M25X_PIVOT_TOURNAMENT) return fail(M25X_EINVAL, "getrf: pivot %d", pivot);
    if (n == 0) return M25X_OK;
    if (n > (1L << 30)) return fail(M25X_EINVAL, "getrf: n too large");
    hipStream_t s = (hipStream_t)stream;
    const bool tp = pivot == M25X_PIVOT_TOURNAMENT;
    int rc;
    if (dtype == M25X_C128)
        rc = tp ? getrf_tp<double2>((double2 *)A, n, lda, ipiv, perm, info, work, wbytes, s)
                : getrf_t<double2>((double2 *)A, n, lda, ipiv, info, work, wbytes, s);
    else if (dtype == M25X_C64)
        rc = tp ? getrf_tp<float2>((float2 *)A, n, lda, ipiv, perm, info, work, wbytes, s)
                : getrf_t<float2>((float2 *)A, n, lda, ipiv, info, work, wbytes, s);
    else
        return fail(M25X_EINVAL, "getrf: dtype %d", dtype);
    if (rc == M25X_OK && perm && !tp) {
        hipLaunchKernelGGL(k_perm, dim3(1), dim3(256), 0, s, (const int *)ipiv, n, perm);
        rc = check_launch("getrf/perm");
    }
    return rc;
}

int m25x_lu_set_lookahead(int on)
{
    if (on != 0 && on != 1) return fail(M25X_EINVAL, "lu_set_lookahead: 0 or 1, not %d", on);
    g_lookahead.store(on, std::memory_order_relaxed);
    return M25X_OK;
}

int m25x_lu_lookahead(void) { return g_lookahead.load(std::memory_order_relaxed); }

size_t m25x_getrs_work_bytes(int dtype, long n, long ldb)
{
    return dtype == M25X_C64 ? getrs_work<float2>(n, ldb) : getrs_work<double2>(n, ldb);
}

int m25x_ipiv_perm(const int *ipiv, long n, int *perm, void *stream)
{
    if (!ipiv || !perm || n < 0) return fail(M25X_EINVAL, "ipiv_perm: bad arguments");
    if (n == 0) return M25X_OK;
    hipLaunchKernelGGL(k_perm, dim3(1), dim3(256), 0, (hipStream_t)stream, ipiv, n, perm);
    return check_launch("ipiv_perm");
}

int m25x_getrs(int dtype, const void *LU, long n, long lda, const int *ipiv, const int *perm, void *B, long ldb,
               int nrhs, int trans, void *work, size_t work_bytes, void *stream)
{
    if (!LU || !ipiv || !B || n < 0 || lda < n) return fail(M25X_EINVAL, "getrs: bad arguments");
    if (n == 0) return M25X_OK;
    hipStream_t s = (hipStream_t)stream;
    if (dtype == M25X_C128)
        return getrs_t<double2>((const double2 *)LU, n, lda, ipiv, perm, (double2 *)B, ldb, nrhs, trans, work,
                                work_bytes, s);
    if (dtype == M25X_C64)
        return getrs_t<float2>((const float2 *)LU, n, lda, ipiv, perm, (float2 *)B, ldb, nrhs, trans, work, work_bytes,
                               s);
    return fail(M25X_EINVAL, "getrs: dtype %d", dtype);
}

}  // extern "C"
