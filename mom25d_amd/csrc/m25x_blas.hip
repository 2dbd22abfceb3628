// m25x_blas.hip - the FP64 kernels of the GMRES refinement: Y = Z X with Z (n x n complex128, row-major) read
// once from HBM per product and X (n x k, k <= 8) staged through LDS in chunks shared by 16 rows; one build per k.
#include <algorithm>
#include "m25x_common.h"

using namespace m25x;

namespace {

constexpr int RK = 8;          // right-hand sides at most
constexpr int CH = 256;        // columns a chunk
constexpr int UJ = CH / 64;    // columns a lane per chunk

// rows a wave: four, two from six right-hand sides on (registers)
template <int K> constexpr int rows_per_wave() { return K <= 5 ? 4 : 2; }

// Each wave takes RPW rows; per chunk of CH columns a lane loads its UJ columns of all RPW rows at once (RPW x UJ
// independent 16 B loads in flight), reads each column's K values of X once from LDS (laid out [K][CH], so a
// wave's reads are consecutive) and applies them to the RPW rows.
// X, Y: leading dimensions ldx, ldy; kk <= K columns in use (the others read as zero and are not written)
template <int K>
__device__ __forceinline__ void zgemm_body(const double2 *__restrict__ Z, long n, long ld,
                                           const double2 *__restrict__ X, long ldx, double2 *__restrict__ Y, long ldy,
                                           int kk, long bx)
{
    constexpr int RPW = rows_per_wave<K>();
    __shared__ double2 xs[K][CH];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const long i0 = bx * (4 * RPW) + wv * RPW;
    double2 acc[RPW][K];
#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
        for (int c = 0; c < K; ++c) acc[r][c] = make_double2(0, 0);
    for (long j0 = 0; j0 < n; j0 += CH) {
        const long jn = n - j0 < CH ? n - j0 : CH;
        // the chunk's Z entries first (from HBM: the long wait), then its X values (K a thread, all in flight
        // before the first is stored to LDS)
        double2 z[RPW][UJ];
#pragma unroll
        for (int r = 0; r < RPW; ++r)
#pragma unroll
            for (int u = 0; u < UJ; ++u) {
                const long jj = lane + 64 * u;
                z[r][u] = (i0 + r < n && jj < jn) ? Z[(i0 + r) * ld + j0 + jj] : make_double2(0, 0);
            }
        double2 xv[CH * K / 256];
#pragma unroll
        for (int it = 0; it < CH * K / 256; ++it) {
            const int idx = tid + it * 256, t = idx / K, c = idx % K;
            xv[it] = (t < jn && c < kk) ? X[(j0 + t) * ldx + c] : make_double2(0, 0);
        }
#pragma unroll
        for (int it = 0; it < CH * K / 256; ++it) {
            const int idx = tid + it * 256;
            xs[idx % K][idx / K] = xv[it];
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < UJ; ++u) {
            double2 x[K];
#pragma unroll
            for (int c = 0; c < K; ++c) x[c] = xs[c][lane + 64 * u];
#pragma unroll
            for (int r = 0; r < RPW; ++r)
#pragma unroll
                for (int c = 0; c < K; ++c) {
                    acc[r][c].x += z[r][u].x * x[c].x - z[r][u].y * x[c].y;
                    acc[r][c].y += z[r][u].x * x[c].y + z[r][u].y * x[c].x;
                }
        }
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
        for (int c = 0; c < K; ++c) {
            double x = acc[r][c].x, y = acc[r][c].y;
            for (int o = 32; o > 0; o >>= 1) { x += __shfl_xor(x, o); y += __shfl_xor(y, o); }
            if (lane == 0 && i0 + r < n && c < kk) Y[(i0 + r) * ldy + c] = make_double2(x, y);
        }
}

template <int K>
__global__ __launch_bounds__(256) void k_zgemm_nk(const double2 *__restrict__ Z, long n, long ld,
                                                  const double2 *__restrict__ X, double2 *__restrict__ Y)
{
    zgemm_body<K>(Z, n, ld, X, K, Y, K, K, blockIdx.x);
}

// one item a grid row (blockIdx.y); row blocks past the item's n leave at once
template <int K>
__global__ __launch_bounds__(256) void k_zgemm_nk_b(const m25x_mv_item *__restrict__ items)
{
    const m25x_mv_item it = items[blockIdx.y];
    if ((long)blockIdx.x * (4 * rows_per_wave<K>()) >= it.n) return;
    zgemm_body<K>((const double2 *)it.Z, it.n, it.ld, (const double2 *)it.X, it.ldx, (double2 *)it.Y, it.ldy, it.k,
                  blockIdx.x);
}

}  // namespace

extern "C" int m25x_zgemm_nk(const double *Z, long n, long ld, const double *X, int k, double *Y, void *stream)
{
    if (!Z || !X || !Y || n < 0 || ld < n || k < 1 || k > RK)
        return fail(M25X_EINVAL, "zgemm_nk: bad arguments (1 <= k <= %d)", RK);
    if (n == 0) return M25X_OK;
    hipStream_t s = (hipStream_t)stream;
    const double2 *Zc = (const double2 *)Z, *Xc = (const double2 *)X;
    double2 *Yc = (double2 *)Y;
    TimedLaunch tl(s, M25X_K_ZGEMM_NK, M25X_C128, 16.0 * n * (double)n + 32.0 * n * k, 8.0 * n * (double)n * k);
    switch (k) {
#define M25X_NK(K)                                                                                            \
    case K:                                                                                                   \
        hipLaunchKernelGGL(k_zgemm_nk<K>, dim3((unsigned)((n + 4 * rows_per_wave<K>() - 1) / (4 * rows_per_wave<K>()))), \
                           dim3(256), 0, s, Zc, n, ld, Xc, Yc);                                                \
        break;
        M25X_NK(1) M25X_NK(2) M25X_NK(3) M25X_NK(4) M25X_NK(5) M25X_NK(6) M25X_NK(7) M25X_NK(8)
#undef M25X_NK
    }
    return check_launch("zgemm_nk");
}

extern "C" int m25x_zgemm_nk_batched(int nitems, const m25x_mv_item *h, const m25x_mv_item *d, void *stream)
{
    if (nitems < 0 || (nitems && (!h || !d))) return fail(M25X_EINVAL, "zgemm_nk_batched: bad arguments");
    long nmax = 0;
    int kmax = 1;
    double bytes = 0, flops = 0;
    for (int i = 0; i < nitems; ++i) {
        const m25x_mv_item &it = h[i];
        if (!it.Z || !it.X || !it.Y || it.n < 0 || it.ld < it.n || it.k < 1 || it.k > RK || it.ldx < it.k ||
            it.ldy < it.k)
            return fail(M25X_EINVAL, "zgemm_nk_batched: item %d: bad arguments (1 <= k <= %d, ld >= n, ldx, ldy >= k)",
                        i, RK);
        nmax = std::max(nmax, it.n);
        kmax = std::max(kmax, it.k);
        bytes += 16.0 * it.n * (double)it.n + 32.0 * it.n * it.k;
        flops += 8.0 * it.n * (double)it.n * it.k;
    }
    if (nitems == 0 || nmax == 0) return M25X_OK;
    hipStream_t s = (hipStream_t)stream;
    TimedLaunch tl(s, M25X_K_ZGEMM_NK, M25X_C128, bytes, flops);
    switch (kmax) {
#define M25X_NKB(K)                                                                                           \
    case K:                                                                                                   \
        hipLaunchKernelGGL(k_zgemm_nk_b<K>, dim3((unsigned)((nmax + 4 * rows_per_wave<K>() - 1) / (4 * rows_per_wave<K>())), \
                                                 (unsigned)nitems), dim3(256), 0, s, d);                      \
        break;
        M25X_NKB(1) M25X_NKB(2) M25X_NKB(3) M25X_NKB(4) M25X_NKB(5) M25X_NKB(6) M25X_NKB(7) M25X_NKB(8)
#undef M25X_NKB
    }
    return check_launch("zgemm_nk_batched");
}

// ---- classical Gram-Schmidt, twice, for the batched GMRES ------------------------------------------------------
// V: (j + 1) basis vectors, each n x k complex128 row-major (vector i at V + i n k); w: n x k. Per column c:
// h1 = V^H w, w1 = w - V h1, h2 = V^H w1, w2 = w1 - V h2, h = h1 + h2, nrm = |w2|, V[j + 1] = w2 / nrm (nrm = 0: w2).
// w1 and w2 go over w, or into V[j + 1] where the caller keeps w (the same reads and writes either way).
// Sums over rows in fixed blocks, then over blocks in a fixed order: the result does not depend on timing.
//
// Four launches, each waiting for the sums of the one before; the basis (3 MB at n = 7799, k = 4, six vectors) stays in
// the caches, so what counts is each launch's chain of memory round trips. Rows are spread so that a thread has one
// up to n k = 32 768 elements (column = the thread's low bits, so reads are consecutive), the basis is read
// GS_CH vectors at a time with the loads in flight together, a wave's GS_CH sums are folded by halving (each exchange
// sends the half that the partner keeps: 8 exchanges for 8 sums over 16 lanes, not 32), and every block of the next
// launch adds the blocks' partial sums itself instead of a launch of one workgroup between them. Seven launches with
// one vector a round trip took 38.5 us at n = 7799, k = 4 on six vectors and 94 on 30, these take 18.1 and 34.2;
// at n = 905 27.9 and 16.6 on six, at n = 20 000 348 and 59 on 30. More than eight columns (many points side by side)
// go in groups of eight, a grid row each, with fewer row blocks as the groups fill the chip by themselves.
namespace {

constexpr int GS_B = 128;                // row blocks at most, and over all groups of columns where each has GS_BMIN
constexpr int GS_BMIN = 16;
constexpr int GS_C = 8;                  // columns a group
constexpr int GS_T = 256;                // threads a block: KP columns x GS_T / KP row lanes
constexpr int GS_MAXV = 64;              // basis vectors at most
constexpr int GS_CH = 8;                 // basis vectors read at a time

constexpr int gs_groups(int k) { return (k + GS_C - 1) / GS_C; }
constexpr int gs_blocks(int k) { return GS_B / gs_groups(k) > GS_BMIN ? GS_B / gs_groups(k) : GS_BMIN; }

// A grid row's columns c0 .. c0 + kc - 1, and its own partial sums (two passes' and the norms').
struct GsGroup {
    int c0, kc;
    long p, q;
};
template <int KP>
__device__ inline GsGroup gs_group(int k)
{
    const int g = blockIdx.y, c0 = g * GS_C;
    return {c0, k - c0 < KP ? k - c0 : KP, (long)g * gridDim.x * GS_MAXV * GS_C, (long)g * gridDim.x * GS_C};
}

// h[i kc + c] = sum over the blocks' partial sums P[b][i kc + c]: m = nv kc entries, up to GS_T / m threads an entry.
__device__ inline void gs_sum(const double2 *__restrict__ P, int nb, int m, double2 *h, double2 *part)
{
    const int t = threadIdx.x, S = m < GS_T ? GS_T / m : 1;
    for (int e0 = 0; e0 < m; e0 += GS_T) {
        const int e = S > 1 ? t % m : e0 + t, sl = S > 1 ? t / m : 0;
        double2 s = make_double2(0, 0);
        if (e < m && sl < S) {
#pragma unroll 8
            for (int b = sl; b < nb; b += S) {
                const double2 p = P[(long)b * m + e];
                s.x += p.x; s.y += p.y;
            }
            if (S > 1) part[t] = s;
            else h[e] = s;
        }
    }
    __syncthreads();
    if (S > 1) {
        if (t < m) {
            double2 s = part[t];
            for (int l = 1; l < S; ++l) { s.x += part[l * m + t].x; s.y += part[l * m + t].y; }
            h[t] = s;
        }
        __syncthreads();
    }
}

// The vectors i0 .. i0 + GS_CH - 1 at element e, the last one repeated past nv (its uses are then dropped or zero).
__device__ inline void gs_load(double2 (&v)[GS_CH], const double2 *__restrict__ V, long nk, long e, int i0, int nv)
{
#pragma unroll
    for (int u = 0; u < GS_CH; ++u) v[u] = V[(long)(i0 + u < nv ? i0 + u : nv - 1) * nk + e];
}

// x - sum_i V[i] h[i] at element e of column c of kc
__device__ inline double2 gs_minus(double2 x, const double2 *__restrict__ V, long nk, long e, int c, int kc, int nv,
                                   const double2 *h)
{
    for (int i0 = 0; i0 < nv; i0 += GS_CH) {
        double2 v[GS_CH];
        gs_load(v, V, nk, e, i0, nv);
#pragma unroll
        for (int u = 0; u < GS_CH; ++u)
            if (i0 + u < nv) {
                const double2 hv = h[(i0 + u) * kc + c];
                x.x -= v[u].x * hv.x - v[u].y * hv.y;
                x.y -= v[u].x * hv.y + v[u].y * hv.x;
            }
    }
    return x;
}

// Partial dots of block blockIdx.x's rows: P[b][i kc + c] = sum_r conj(V[i][r][c]) w[r][c]. UPD: of x = w - V h, h the
// sum of the last pass's partial sums Pin, x stored (it may be w); block 0 stores h to H.
template <int KP, bool UPD>
__global__ __launch_bounds__(GS_T) void k_gs_dots(const double2 *__restrict__ V, long n, int k, int nv, const double2 *w,
                                                 double2 *x, const double2 *__restrict__ Pin,
                                                 double2 *__restrict__ H, double2 *__restrict__ P)
{
    __shared__ double2 red[GS_MAXV][GS_T / 64][KP];
    __shared__ double2 h[UPD ? GS_MAXV * KP : 1], part[UPD ? GS_T : 1];
    constexpr int RL = GS_T / KP;
    const int t = threadIdx.x, c = t % KP, rl = t / KP, wv = t >> 6, lane = t & 63;
    const GsGroup g = gs_group<KP>(k);
    const int kc = g.kc, m = nv * kc;
    const long nk = n * k, step = (long)gridDim.x * RL;
    V += g.c0;
    w += g.c0;
    x += g.c0;
    if (UPD) {
        gs_sum(Pin + g.p, gridDim.x, m, h, part);
        if (blockIdx.x == 0)
            for (int e = t; e < m; e += GS_T) H[e / kc * k + g.c0 + e % kc] = h[e];
        if (c < kc)                              // each thread updates the elements it reads below
            for (long r = (long)blockIdx.x * RL + rl; r < n; r += step)
                x[r * k + c] = gs_minus(w[r * k + c], V, nk, r * k + c, c, kc, nv, h);
    }
    for (int i0 = 0; i0 < nv; i0 += GS_CH) {
        double2 a[GS_CH];
#pragma unroll
        for (int u = 0; u < GS_CH; ++u) a[u] = make_double2(0, 0);
        if (c < kc)
            for (long r = (long)blockIdx.x * RL + rl; r < n; r += step) {
                const double2 xv = UPD ? x[r * k + c] : w[r * k + c];
                double2 v[GS_CH];
                gs_load(v, V, nk, r * k + c, i0, nv);
#pragma unroll
                for (int u = 0; u < GS_CH; ++u) {
                    a[u].x += v[u].x * xv.x + v[u].y * xv.y;
                    a[u].y += v[u].x * xv.y - v[u].y * xv.x;
                }
            }
        // the wave's row lanes: three halvings leave one sum a lane, vector 4 b0 + 2 b1 + b2 of its row lane's low bits
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            const int half = 4 >> s, o = KP << s;
            const bool up = lane & o;
#pragma unroll
            for (int u = 0; u < half; ++u) {
                const double2 keep = up ? a[u + half] : a[u], send = up ? a[u] : a[u + half];
                a[u].x = keep.x + __shfl_xor(send.x, o);
                a[u].y = keep.y + __shfl_xor(send.y, o);
            }
        }
#pragma unroll
        for (int o = KP << 3; o < 64; o <<= 1) { a[0].x += __shfl_xor(a[0].x, o); a[0].y += __shfl_xor(a[0].y, o); }
        const int b = lane / KP, i = i0 + ((b & 1) << 2 | (b & 2) | (b >> 2 & 1));
        if (lane < 8 * KP && i < nv) red[i][wv][c] = a[0];
    }
    __syncthreads();
    for (int e = t; e < m; e += GS_T) {
        const double2 *q = &red[e / kc][0][e % kc];
        double2 s = q[0];
#pragma unroll
        for (int w = 1; w < GS_T / 64; ++w) { s.x += q[w * KP].x; s.y += q[w * KP].y; }
        P[g.p + (long)blockIdx.x * m + e] = s;
    }
}

// x -= V h2, h2 the sum of the partial sums Pin; Q[b][c] = partial |x|^2; block 0 adds h2 to H.
template <int KP>
__global__ __launch_bounds__(GS_T) void k_gs_final(const double2 *__restrict__ V, long n, int k, int nv,
                                                  double2 *__restrict__ x, const double2 *__restrict__ Pin,
                                                  double2 *__restrict__ H, double *__restrict__ Q)
{
    __shared__ double2 h[GS_MAXV * KP], part[GS_T];
    __shared__ double red[GS_T / 64][KP];
    constexpr int RL = GS_T / KP;
    const int t = threadIdx.x, c = t % KP, rl = t / KP;
    const GsGroup g = gs_group<KP>(k);
    const int kc = g.kc, m = nv * kc;
    V += g.c0;
    x += g.c0;
    gs_sum(Pin + g.p, gridDim.x, m, h, part);
    if (blockIdx.x == 0)
        for (int e = t; e < m; e += GS_T) {
            double2 &to = H[e / kc * k + g.c0 + e % kc];
            to.x += h[e].x; to.y += h[e].y;
        }
    double q = 0;
    if (c < kc)
        for (long r = (long)blockIdx.x * RL + rl; r < n; r += (long)gridDim.x * RL) {
            const double2 xv = gs_minus(x[r * k + c], V, n * k, r * k + c, c, kc, nv, h);
            x[r * k + c] = xv;
            q += xv.x * xv.x + xv.y * xv.y;
        }
#pragma unroll
    for (int o = KP; o < 64; o <<= 1) q += __shfl_xor(q, o);
    if ((t & 63) < KP) red[t >> 6][c] = q;
    __syncthreads();
    if (t < kc) {
        double s = red[0][t];
        for (int w = 1; w < GS_T / 64; ++w) s += red[w][t];
        Q[g.q + blockIdx.x * KP + t] = s;
    }
}

// H[nv][c] = |x| (real, block 0), out = x / |x| (out may be x); Q: nb blocks' partial |x|^2.
template <int KP>
__global__ __launch_bounds__(GS_T) void k_gs_scale(const double2 *x, long n, int k, int nv, int nb,
                                                  const double *__restrict__ Q, double2 *__restrict__ H, double2 *out)
{
    __shared__ double red[GS_T / 64][KP];
    constexpr int RL = GS_T / KP;
    const int t = threadIdx.x, c = t % KP, rl = t / KP;
    const long r = (long)blockIdx.x * RL + rl;
    const int c0 = blockIdx.y * GS_C, kc = k - c0 < KP ? k - c0 : KP;
    const bool in = c < kc && r < n;
    const double2 xv = in ? x[r * k + c0 + c] : make_double2(0, 0);
    double q = 0;
    if (c < kc)
        for (int b = rl; b < nb; b += RL) q += Q[(long)blockIdx.y * nb * GS_C + b * KP + c];
#pragma unroll
    for (int o = KP; o < 64; o <<= 1) q += __shfl_xor(q, o);
    if ((t & 63) < KP) red[t >> 6][c] = q;
    __syncthreads();
    double s = red[0][c];
    for (int w = 1; w < GS_T / 64; ++w) s += red[w][c];
    const double nr = sqrt(s), sc = nr > 0 ? 1.0 / nr : 1.0;
    if (blockIdx.x == 0 && t < kc) H[nv * k + c0 + t] = make_double2(nr, 0);
    if (in) out[r * k + c0 + c] = make_double2(xv.x * sc, xv.y * sc);
}

template <int KP>
void cgs2(const double2 *V, long n, int k, int nv, const double2 *w, double2 *x, double2 *H, double2 *out, double2 *P,
          hipStream_t s)
{
    const int ng = gs_groups(k);
    const long full = (n + GS_T / KP - 1) / (GS_T / KP);
    const int nb = (int)std::min<long>(full, gs_blocks(k));
    double2 *P2 = P + (size_t)ng * nb * GS_MAXV * GS_C;
    double *Q = (double *)(P2 + (size_t)ng * nb * GS_MAXV * GS_C);
    hipLaunchKernelGGL((k_gs_dots<KP, false>), dim3(nb, ng), dim3(GS_T), 0, s, V, n, k, nv, w, x, (const double2 *)nullptr,
                       (double2 *)nullptr, P);
    hipLaunchKernelGGL((k_gs_dots<KP, true>), dim3(nb, ng), dim3(GS_T), 0, s, V, n, k, nv, w, x, (const double2 *)P, H, P2);
    hipLaunchKernelGGL(k_gs_final<KP>, dim3(nb, ng), dim3(GS_T), 0, s, V, n, k, nv, x, (const double2 *)P2, H, Q);
    hipLaunchKernelGGL(k_gs_scale<KP>, dim3((unsigned)full, ng), dim3(GS_T), 0, s, (const double2 *)x, n, k, nv, nb,
                       (const double *)Q, H, out);
}

// x: where w1 and w2 go, w or vnext
int cgs2_any(const char *who, int kmax, const double *V, long n, int k, int nv, const double *w, double *x, double *hcol,
             double *vnext, void *work, size_t work_bytes, size_t need, hipStream_t s)
{
    if (!V || !w || !hcol || !vnext || !work || n < 1 || k < 1 || k > kmax || nv < 1 || nv > GS_MAXV - 1)
        return fail(M25X_EINVAL, "%s: bad arguments (1 <= k <= %d, 1 <= nv <= %d)", who, kmax, GS_MAXV - 1);
    if (work_bytes < need) return fail(M25X_EINVAL, "%s: workspace too small", who);
    TimedLaunch tl(s, M25X_K_CGS2, M25X_C128, 16.0 * n * k * (2.0 * nv + 3), 16.0 * n * k * nv);
    const auto run = k == 1 ? cgs2<1> : k == 2 ? cgs2<2> : k <= 4 ? cgs2<4> : cgs2<8>;
    run((const double2 *)V, n, k, nv, (const double2 *)w, (double2 *)x, (double2 *)hcol, (double2 *)vnext, (double2 *)work, s);
    return check_launch(who);
}

}  // namespace

extern "C" size_t m25x_cgs2_cols_work_bytes(int k)
{
    if (k < 1 || k > M25X_CGS2_COLS) return 0;
    return (size_t)gs_groups(k) * gs_blocks(k) * GS_C * (2 * GS_MAXV * sizeof(double2) + sizeof(double));
}

extern "C" size_t m25x_cgs2_work_bytes(void) { return m25x_cgs2_cols_work_bytes(GS_C); }

extern "C" int m25x_cgs2(const double *V, long n, int k, int nv, double *w, double *hcol, double *vnext, void *work,
                         size_t work_bytes, void *stream)
{
    return cgs2_any("cgs2", GS_C, V, n, k, nv, w, w, hcol, vnext, work, work_bytes, m25x_cgs2_work_bytes(),
                    (hipStream_t)stream);
}

extern "C" int m25x_cgs2_cols(const double *V, long n, int k, int nv, double *w, double *hcol, double *vnext, void *work,
                              size_t work_bytes, void *stream)
{
    return cgs2_any("cgs2_cols", M25X_CGS2_COLS, V, n, k, nv, w, w, hcol, vnext, work, work_bytes,
                    m25x_cgs2_cols_work_bytes(k), (hipStream_t)stream);
}

extern "C" int m25x_cgs2_keep(const double *V, long n, int k, int nv, const double *w, double *hcol, double *vnext,
                              void *work, size_t work_bytes, void *stream)
{
    return cgs2_any("cgs2_keep", M25X_CGS2_COLS, V, n, k, nv, w, vnext, hcol, vnext, work, work_bytes,
                    m25x_cgs2_cols_work_bytes(k), (hipStream_t)stream);
}

// ---- the solves' right-hand sides between precisions ----------------------------------------------------------
// dst[i][c] = r[i] src[i][c], computed in FP64 and rounded once to dst's type: one pass in place of a product, a
// conversion and a copy (each a launch of 9-12 us for a matter of 0.5 MB; a complex64 solve of four right-hand sides at
// n = 7799 433 -> 417 us with its conversions). A thread an element, columns fastest.
namespace {

template <typename S, typename D>
__global__ void k_cast_rows(const S *__restrict__ src, long lds, D *__restrict__ dst, long ldd, long n, long k,
                            const double *__restrict__ r)
{
    const long idx = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (idx >= n * k) return;
    const long i = idx / k, c = idx % k;
    const S v = src[i * lds + c];
    double x = v.x, y = v.y;
    if (r) { x *= r[i]; y *= r[i]; }
    dst[i * ldd + c] = D{(decltype(D::x))x, (decltype(D::x))y};
}

template <typename S, typename D>
void cast_rows(const void *src, long lds, void *dst, long ldd, long n, long k, const double *r, hipStream_t s)
{
    hipLaunchKernelGGL((k_cast_rows<S, D>), dim3((unsigned)((n * k + 255) / 256)), dim3(256), 0, s, (const S *)src, lds,
                       (D *)dst, ldd, n, k, r);
}

}  // namespace

extern "C" int m25x_cast_rows(int src_dtype, const void *src, long lds, int dst_dtype, void *dst, long ldd, long n,
                              long k, const double *r, void *stream)
{
    const auto known = [](int d) { return d == M25X_C64 || d == M25X_C128; };
    if (!known(src_dtype) || !known(dst_dtype) || n < 0 || k < 0 || (n > 0 && k > (1L << 38) / n) ||
        (n > 0 && k > 0 && (!src || !dst || lds < k || ldd < k)))
        return fail(M25X_EINVAL, "cast_rows: bad arguments");
    if (n == 0 || k == 0) return M25X_OK;
    hipStream_t s = (hipStream_t)stream;
    if (src_dtype == M25X_C128) {
        if (dst_dtype == M25X_C128) cast_rows<double2, double2>(src, lds, dst, ldd, n, k, r, s);
        else cast_rows<double2, float2>(src, lds, dst, ldd, n, k, r, s);
    } else {
        if (dst_dtype == M25X_C128) cast_rows<float2, double2>(src, lds, dst, ldd, n, k, r, s);
        else cast_rows<float2, float2>(src, lds, dst, ldd, n, k, r, s);
    }
    return check_launch("cast_rows");
}
