// m25x_fill.hip - the impedance-matrix fill on gfx950: far field (centroid rule) in symmetric 32 x 32 tiles,
// the near-field correction as per-pair moments plus a deterministic per-entry gather, the via fan and radial
// sums, the Sommerfeld-Hankel transforms of the Green's tables, the near-pair search and the equilibration.
//
// Everything is FP64 (complex128); only the fill's store may narrow to complex64. The far fill is bound by its
// Z stores (16 B an entry, each tile written once and its mirror once through LDS); the kernel values come from
// the tables, read through L2 (a table is 8192 x 32 B).
#include "m25x_common.h"

#include <type_traits>

using namespace m25x;

namespace {

struct DMesh {
    int Ne, Nt;
    const int *ep, *em, *lt, *te;
    const double *ap, *am, *vp, *vm, *cent, *area, *ta, *tv;
};

DMesh dmesh(const m25x_mesh *g)
{
    DMesh m;
    m.Ne = g->Ne; m.Nt = g->Nt;
    m.ep = g->ep; m.em = g->em; m.lt = g->lt; m.te = g->te;
    m.ap = g->ap; m.am = g->am; m.vp = g->vp; m.vm = g->vm; m.cent = g->cent; m.area = g->area;
    m.ta = g->ta; m.tv = g->tv;
    return m;
}

__device__ inline double cdist(const double *c, int p, int q)
{
    double dx = c[2 * p] - c[2 * q], dy = c[2 * p + 1] - c[2 * q + 1];
    return sqrt(dx * dx + dy * dy);
}

template <typename T> __device__ inline void store_c(T *Z, size_t i, double2 v);
template <> __device__ inline void store_c<double2>(double2 *Z, size_t i, double2 v) { Z[i] = v; }
template <> __device__ inline void store_c<float2>(float2 *Z, size_t i, double2 v)
{
    Z[i] = make_float2((float)v.x, (float)v.y);
}

// ---- far field -------------------------------------------------------------------------------------------
// One 512-thread workgroup per 32 x 32 tile of edge pairs in the upper triangle (tile row <= tile column):
// Z[m, n] for m in the row tile, n in the column tile, each the reference's sum over the halves (s, t) of
//   a_ms a_nt [jw (c_ms - v_ms).(c_nt - v_nt) G_A(r) + 4 G_q(r) / (jw)],  r = |c_ms - c_nt|,
// (mom25d_core.cpp:152-170), stored at (m, n) and, through LDS, at (n, m): Z is symmetric bit for bit.
//
// The kernel's value (square roots, divisions, two interpolations) bounds the fill, and it depends on the two triangles
// only: edges that follow each other share triangles (32 edges of a mesh have some 33, not 64), so it is computed once
// for each pair of the tile's triangles and the entries read it from LDS: a quarter of the evaluations, 7799 unknowns
// 1130 -> 580 us. Where a tile's triangles are too many for the LDS (edges in an order of their own) each entry
// computes its own four.
struct Half {
    double a, dx, dy, cx, cy;
    int lay, tri;
};

constexpr int FT = 32, FTH = 512;         // edges of a tile's side; threads
constexpr int FP = 1296;                  // triangle pairs that the LDS holds (36 x 36; two workgroups a CU)

template <typename TZ>
__global__ __launch_bounds__(FTH) void k_fill_far(TZ *__restrict__ Z, long ld, DMesh g, DTab T, double w)
{
    const int ti = blockIdx.y, tj = blockIdx.x;
    if (ti > tj) return;
    __shared__ Half hf[2][2 * FT];                           // [rows, columns][s * 32 + edge]
    __shared__ __align__(16) int tr[2][2 * FT];              // their triangles
    __shared__ double2 tile[FT][FT + 1];
    __shared__ double2 KA[FP], KQ[FP];                       // G_A and G_q of a pair of distinct triangles
    __shared__ unsigned char un[2][2 * FT], rep[2][2 * FT];  // a half's number among its side's distinct triangles, and
    __shared__ unsigned short firsts[2][4];                  // a distinct triangle's first half; which halves are first
    const int tid = threadIdx.x;
    const int m0 = ti * FT, n0 = tj * FT, Ne = g.Ne;
    if (tid < 4 * FT) {
        const int side = tid / (2 * FT), k = tid % (2 * FT), s = k / FT, e = k % FT;
        const int edge = (side ? n0 : m0) + e;
        Half h;
        h.a = h.dx = h.dy = h.cx = h.cy = 0.0;
        h.lay = 0; h.tri = -1;
        if (edge < Ne) {
            const int tri = s ? g.em[edge] : g.ep[edge];
            const double alpha = s ? g.am[edge] : g.ap[edge];
            const double *v = (s ? g.vm : g.vp) + 2 * (size_t)edge;
            h.a = alpha * g.area[tri];
            h.cx = g.cent[2 * tri]; h.cy = g.cent[2 * tri + 1];
            h.dx = h.cx - v[0]; h.dy = h.cy - v[1];
            h.lay = g.lt[tri];
            h.tri = tri;
        }
        hf[side][k] = h;
        tr[side][k] = h.tri;
    }
    __syncthreads();
    // the distinct triangles of each side: four lanes a half look for the first half with its triangle
    const int side = tid >> 8, q = tid & 3, half = (tid >> 2) & 63;
    int first = half;
    {
        const int mine = tr[side][half];
        const int4 *t4 = (const int4 *)tr[side] + 4 * q;
#pragma unroll
        for (int i = 3; i >= 0; --i) {
            const int4 v = t4[i];
            const int b = 16 * q + 4 * i;
            if (v.w == mine) first = min(first, b + 3);
            if (v.z == mine) first = min(first, b + 2);
            if (v.y == mine) first = min(first, b + 1);
            if (v.x == mine) first = min(first, b);
        }
        first = min(first, __builtin_amdgcn_update_dpp(first, first, 0xB1, 0xF, 0xF, false));      // over the quad
        first = min(first, __builtin_amdgcn_update_dpp(first, first, 0x4E, 0xF, 0xF, false));
    }
    {
        // a wave holds 16 halves, four lanes each: one bit a half
        unsigned long long m = __builtin_amdgcn_ballot_w64(first == half && q == 0) & 0x1111111111111111ull;
        m = (m | m >> 3) & 0x0303030303030303ull;
        m = (m | m >> 6) & 0x000f000f000f000full;
        m = (m | m >> 12) & 0x000000ff000000ffull;
        m = (m | m >> 24) & 0xffffull;
        if ((tid & 63) == 0) firsts[side][(tid >> 6) & 3] = (unsigned short)m;
    }
    __syncthreads();
    unsigned long long fm[2];
#pragma unroll
    for (int d = 0; d < 2; ++d)
        fm[d] = (unsigned long long)firsts[d][0] | (unsigned long long)firsts[d][1] << 16 |
                (unsigned long long)firsts[d][2] << 32 | (unsigned long long)firsts[d][3] << 48;
    if (q == 0) {
        const int u = __popcll(fm[side] & ((1ull << first) - 1));
        un[side][half] = (unsigned char)u;
        if (first == half) rep[side][u] = (unsigned char)half;
    }
    __syncthreads();
    const int ncol = __popcll(fm[1]), np = __popcll(fm[0]) * ncol;
    const bool shared = np <= FP;
    if (shared) {
        for (int p = tid; p < np; p += FTH) {
            const int a = p / ncol;
            const Half &hm = hf[0][rep[0][a]], &hn = hf[1][rep[1][p - a * ncol]];
            const double ddx = hm.cx - hn.cx, ddy = hm.cy - hn.cy;
            double2 ga, gq;
            tab_kern(T, hm.lay, hn.lay, sqrt(ddx * ddx + ddy * ddy), ga, gq);
            KA[p] = ga;
            KQ[p] = gq;
        }
        __syncthreads();
    }
    const int c = tid % FT, rg = tid / FT;          // rows rg and rg + 16
    const double iw = 1.0 / w;
    const Half cn0 = hf[1][c], cn1 = hf[1][FT + c];
    const int u0 = un[1][c], u1 = un[1][FT + c];
#pragma unroll
    for (int k = 0; k < FT * FT / FTH; ++k) {
        const int r = rg + FTH / FT * k;
        double vx = 0.0, vy = 0.0;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const Half hm = hf[0][s * FT + r];
            const int pr = un[0][s * FT + r] * ncol;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const Half &hn = t ? cn1 : cn0;
                double2 ga, gq;
                if (shared) {
                    const int p = pr + (t ? u1 : u0);
                    ga = KA[p];
                    gq = KQ[p];
                } else {
                    const double ddx = hm.cx - hn.cx, ddy = hm.cy - hn.cy;
                    tab_kern(T, hm.lay, hn.lay, sqrt(ddx * ddx + ddy * ddy), ga, gq);
                }
                const double wd = w * (hm.dx * hn.dx + hm.dy * hn.dy);
                const double tx = -wd * ga.y + 4.0 * gq.y * iw, ty = wd * ga.x - 4.0 * gq.x * iw;
                const double f = hm.a * hn.a;
                vx += f * tx; vy += f * ty;
            }
        }
        tile[r][c] = make_double2(vx, vy);
    }
    __syncthreads();
    const bool diag = ti == tj;
#pragma unroll
    for (int k = 0; k < FT * FT / FTH; ++k) {
        const int r = rg + FTH / FT * k, m = m0 + r, n = n0 + c;
        if (m < Ne && n < Ne) store_c(Z, (size_t)m * ld + n, (diag && r > c) ? tile[c][r] : tile[r][c]);
    }
    if (!diag) {
#pragma unroll
        for (int k = 0; k < FT * FT / FTH; ++k) {
            const int r = rg + FTH / FT * k, n = n0 + r, m = m0 + c;
            if (n < Ne && m < Ne) store_c(Z, (size_t)n * ld + m, tile[c][r]);
        }
    }
}

// far field of arbitrary row / column edge lists, one thread an entry (mom25d_core.cpp:176-211)
__global__ void k_far_block(const int *R, int nr, const int *C, int nc, DMesh g, DTab T, double w, double2 *o)
{
    const long idx = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (idx >= (long)nr * nc) return;
    const int i = (int)(idx / nc), j = (int)(idx % nc);
    const int m = R[i], n = C[j];
    const int pm[2] = {g.ep[m], g.em[m]}, pn[2] = {g.ep[n], g.em[n]};
    const double am_[2] = {g.ap[m] * g.area[pm[0]], g.am[m] * g.area[pm[1]]};
    const double an[2] = {g.ap[n] * g.area[pn[0]], g.am[n] * g.area[pn[1]]};
    const double dx[2] = {g.cent[2 * pm[0]] - g.vp[2 * m], g.cent[2 * pm[1]] - g.vm[2 * m]};
    const double dy[2] = {g.cent[2 * pm[0] + 1] - g.vp[2 * m + 1], g.cent[2 * pm[1] + 1] - g.vm[2 * m + 1]};
    const double ex[2] = {g.cent[2 * pn[0]] - g.vp[2 * n], g.cent[2 * pn[1]] - g.vm[2 * n]};
    const double ey[2] = {g.cent[2 * pn[0] + 1] - g.vp[2 * n + 1], g.cent[2 * pn[1] + 1] - g.vm[2 * n + 1]};
    const double iw = 1.0 / w;
    double vx = 0, vy = 0;
    for (int s = 0; s < 2; ++s)
        for (int t = 0; t < 2; ++t) {
            double2 ga, gq;
            tab_kern(T, g.lt[pm[s]], g.lt[pn[t]], cdist(g.cent, pm[s], pn[t]), ga, gq);
            const double wd = w * (dx[s] * ex[t] + dy[s] * ey[t]);
            const double f = am_[s] * an[t];
            vx += f * (-wd * ga.y + 4.0 * gq.y * iw);
            vy += f * (wd * ga.x - 4.0 * gq.x * iw);
        }
    o[idx] = make_double2(vx, vy);
}

// ---- near field ------------------------------------------------------------------------------------------
// the rule over the smaller triangle of a pair, ties by index (mom25d_core.cpp:321-324)
__device__ inline bool rule_over_p(double ap, double aq, int p, int q)
{
    const double tie = 1e-9 * fmax(ap, aq);
    return fabs(ap - aq) <= tie ? p <= q : ap < aq;
}

// analytic inner integral of 1/sqrt(rho^2 + d^2) over triangle V, 6-point outer rule (mom25d_core.cpp:331-365)
__device__ void offplane_one(const double *V, const double *P6, const double *W6, double d, double &m0,
                             double mro[2], double mrs[2], double &mrr)
{
    const double ad = fabs(d);
    double L[3], tau[3][2], un[3][2];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int j = (i + 1) % 3;
        const double ex = V[2 * j] - V[2 * i], ey = V[2 * j + 1] - V[2 * i + 1];
        L[i] = sqrt(ex * ex + ey * ey);
        tau[i][0] = ex / L[i]; tau[i][1] = ey / L[i];
        un[i][0] = tau[i][1]; un[i][1] = -tau[i][0];
    }
    m0 = 0; mro[0] = mro[1] = 0; mrs[0] = mrs[1] = 0; mrr = 0;
    for (int k = 0; k < 6; ++k) {
        const double rx = P6[2 * k], ry = P6[2 * k + 1], wq = W6[k];
        double I1 = 0, IRx = 0, IRy = 0;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const double dvx = V[2 * i] - rx, dvy = V[2 * i + 1] - ry;
            const double sm = dvx * tau[i][0] + dvy * tau[i][1];
            const double sp = sm + L[i];
            const double t0 = dvx * un[i][0] + dvy * un[i][1];
            const double R02 = t0 * t0 + d * d, R0 = sqrt(R02);
            const double Rm = sqrt(R02 + sm * sm), Rp = sqrt(R02 + sp * sp);
            const double lg = (R0 > 1e-14 * L[i]) ? asinh(sp / R0) - asinh(sm / R0) : 0.0;
            const double beta = atan2(t0 * sp, R02 + ad * Rp) - atan2(t0 * sm, R02 + ad * Rm);
            I1 += t0 * lg - ad * beta;
            const double eR = 0.5 * (R02 * lg + sp * Rp - sm * Rm);
            IRx += eR * un[i][0]; IRy += eR * un[i][1];
        }
        const double Wx = IRx + rx * I1, Wy = IRy + ry * I1;
        m0 += wq * I1;
        mro[0] += wq * rx * I1; mro[1] += wq * ry * I1;
        mrs[0] += wq * Wx; mrs[1] += wq * Wy;
        mrr += wq * (rx * Wx + ry * Wy);
    }
}

struct DQuad {
    const double *nodes;
    const int *tris;
    const double *P3, *W3, *P6, *W6;
};

// The separations of the parts extracted from table t, at most two, and their coefficients
__device__ __forceinline__ int extracted(const DTab &T, int t, double (&d)[2], double2 (&cA)[2], double2 (&cq)[2])
{
    d[0] = d[1] = 0;
    const int kd = T.kind[t];
    if (kd == 0) {
        cA[0] = T.cA[t]; cq[0] = T.cq[t];
        if (!(T.dimg[t] > 0)) return 1;
        d[1] = T.dimg[t]; cA[1] = T.cAi[t]; cq[1] = T.cqi[t];
        return 2;
    }
    if (kd != 1) return 0;
    d[0] = T.d[t]; cA[0] = T.cA[t]; cq[0] = T.cq[t];
    return 1;
}
// the six moments of an extracted part at separation d of the pair (p, q)
__device__ void static_part(const DMesh &g, const DQuad &qd, int p, int q, double d, double (&m)[6])
{
    const bool keep = rule_over_p(g.area[p], g.area[q], p, q);
    const int po = keep ? p : q, qi = keep ? q : p;
    double V[6];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int nd = qd.tris[3 * qi + j];
        V[2 * j] = qd.nodes[2 * nd]; V[2 * j + 1] = qd.nodes[2 * nd + 1];
    }
    double mo[2], ms[2];
    offplane_one(V, qd.P6 + 12 * (size_t)po, qd.W6 + 6 * (size_t)po, d, m[0], mo, ms, m[5]);
    m[1] = keep ? mo[0] : ms[0]; m[2] = keep ? mo[1] : ms[1];
    m[3] = keep ? ms[0] : mo[0]; m[4] = keep ? ms[1] : mo[1];
}
// stat: the extracted parts' moments of every pair (geometry and separations only), 2 x 6 doubles
__global__ __launch_bounds__(256) void k_near_static(DMesh g, DTab T, DQuad qd, const int *P, const int *Q, long n,
                                                     double *stat)
{
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int p = P[i], q = Q[i];
    double d[2], m[6];
    double2 cA[2], cq[2];
    const int next = extracted(T, T.tab[g.lt[p] * T.L + g.lt[q]], d, cA, cq);
    for (int k = 0; k < next; ++k) {
        static_part(g, qd, p, q, d[k], m);
#pragma unroll
        for (int j = 0; j < 6; ++j) stat[12 * (size_t)i + 6 * k + j] = m[j];
    }
}

// One thread a near pair: the smooth rest by 3 x 3 (same interface) or 6 x 6 (cross) quadrature, the extracted
// parts analytically (KEPT: from stat, k_near_static's, kept across frequencies), less the centroid value the far fill
// put there (mom25d_core.cpp:417-476). M: n x 7 complex128 (M0, Mox, Moy, Msx, Msy, Mrr, Mq). The lookups' latency
// bounds it: with the analytic parts in this kernel a thread had 194 registers, two waves a SIMD, and its lookups
// came one at a time. 1.5 million pairs (7799 unknowns): 345 -> 259 us with the
// caches warm.
template <bool KEPT>
__global__ __launch_bounds__(256, KEPT ? 4 : 2) void k_near_moments(DMesh g, DTab T, DQuad qd, const int *P, const int *Q, long n,
                                                      const double *stat, double2 *M, double2 *qcorr)
{
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int p = P[i], q = Q[i];
    const int la = g.lt[p], lb = g.lt[q];
    const int t = T.tab[la * T.L + lb];
    double2 M0 = {0, 0}, Mox = {0, 0}, Moy = {0, 0}, Msx = {0, 0}, Msy = {0, 0}, Mrr = {0, 0}, Mq = {0, 0};
    auto smooth = [&](auto npc, const double *Pp, const double *Wp) __attribute__((always_inline)) {
        constexpr int np = decltype(npc)::value;
        double qx[np], qy[np], qw[np];
#pragma unroll
        for (int b = 0; b < np; ++b) {
            qx[b] = Pp[2 * np * (size_t)q + 2 * b];
            qy[b] = Pp[2 * np * (size_t)q + 2 * b + 1];
            qw[b] = Wp[np * (size_t)q + b];
        }
#pragma unroll 1
        for (int a = 0; a < np; ++a) {
            const double pax = Pp[2 * np * (size_t)p + 2 * a], pay = Pp[2 * np * (size_t)p + 2 * a + 1];
            const double wa = Wp[np * (size_t)p + a];
#pragma unroll
            for (int b0 = 0; b0 < np; b0 += 3) {
                double2 ga[3], gq[3];                // three lookups in flight before the first is used
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    const double dx = pax - qx[b0 + b], dy = pay - qy[b0 + b];
                    tab_rest(T, t, sqrt(dx * dx + dy * dy), ga[b], gq[b]);
                }
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    const double wt = wa * qw[b0 + b], x = qx[b0 + b], y = qy[b0 + b];
                    const double2 A = cscale(ga[b], wt);
                    M0 = cadd(M0, A);
                    Mox = cadd(Mox, cscale(A, pax)); Moy = cadd(Moy, cscale(A, pay));
                    Msx = cadd(Msx, cscale(A, x)); Msy = cadd(Msy, cscale(A, y));
                    Mrr = cadd(Mrr, cscale(A, pax * x + pay * y));
                    Mq = cadd(Mq, cscale(gq[b], wt));
                }
            }
        }
    };
    if (la == lb) smooth(std::integral_constant<int, 3>{}, qd.P3, qd.W3);
    else smooth(std::integral_constant<int, 6>{}, qd.P6, qd.W6);
    double dd[2];
    double2 cAs[2], cqs[2];
    const int next = extracted(T, t, dd, cAs, cqs);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        if (k >= next) break;
        double m[6];
        if constexpr (KEPT) {
#pragma unroll
            for (int j = 0; j < 6; ++j) m[j] = stat[12 * (size_t)i + 6 * k + j];
        } else {
            static_part(g, qd, p, q, dd[k], m);
        }
        const double2 cA = cAs[k], cq = cqs[k];
        M0 = cadd(M0, cscale(cA, m[0])); Mox = cadd(Mox, cscale(cA, m[1])); Moy = cadd(Moy, cscale(cA, m[2]));
        Msx = cadd(Msx, cscale(cA, m[3])); Msy = cadd(Msy, cscale(cA, m[4])); Mrr = cadd(Mrr, cscale(cA, m[5]));
        Mq = cadd(Mq, cscale(cq, m[0]));
    }
    {
        const double r = cdist(g.cent, p, q);
        double2 ga, gq;
        tab_kern(T, la, lb, r, ga, gq);
        const double wgt = g.area[p] * g.area[q];
        const double cpx = g.cent[2 * p], cpy = g.cent[2 * p + 1], cqx = g.cent[2 * q], cqy = g.cent[2 * q + 1];
        ga = cscale(ga, wgt); gq = cscale(gq, wgt);
        M0 = csub(M0, ga);
        Mox = csub(Mox, cscale(ga, cpx)); Moy = csub(Moy, cscale(ga, cpy));
        Msx = csub(Msx, cscale(ga, cqx)); Msy = csub(Msy, cscale(ga, cqy));
        Mrr = csub(Mrr, cscale(ga, cpx * cqx + cpy * cqy));
        Mq = csub(Mq, gq);
    }
    double2 *o = M + 7 * (size_t)i;
    o[0] = M0; o[1] = Mox; o[2] = Moy; o[3] = Msx; o[4] = Msy; o[5] = Mrr; o[6] = Mq;
    if (qcorr) qcorr[i] = Mq;
}

// a pair's value for edge slots s (of p) and u (of q) (mom25d_core.cpp:483-488)
__device__ inline double2 slot_value(const DMesh &g, int p, int q, int s, int u, const double2 *Mi, double w,
                                     double iw)
{
    const double am_ = g.ta[3 * p + s], vx = g.tv[6 * p + 2 * s], vy = g.tv[6 * p + 2 * s + 1];
    const double an = g.ta[3 * q + u], wx = g.tv[6 * q + 2 * u], wy = g.tv[6 * q + 2 * u + 1];
    const double2 M0 = Mi[0], Mox = Mi[1], Moy = Mi[2], Msx = Mi[3], Msy = Mi[4], Mrr = Mi[5], Mq = Mi[6];
    const double vw = vx * wx + vy * wy;
    const double2 Ac = make_double2(Mrr.x - (wx * Mox.x + wy * Moy.x) - (vx * Msx.x + vy * Msy.x) + vw * M0.x,
                                    Mrr.y - (wx * Mox.y + wy * Moy.y) - (vx * Msx.y + vy * Msy.y) + vw * M0.y);
    // jw Ac + 4 Mq / (jw)
    const double2 t = make_double2(-w * Ac.y + 4.0 * Mq.y * iw, w * Ac.x - 4.0 * Mq.x * iw);
    return cscale(t, am_ * an);
}

// one thread a near entry: its contributions summed in a fixed order, then added to Z once
template <typename TZ>
__global__ __launch_bounds__(256) void k_near_scatter(TZ *Z, long ld, DMesh g, const int *P, const int *Q,
                                                      const double2 *M, long nentry, const int *erow,
                                                      const int *ecol, const int *estart, const int *contrib,
                                                      double w)
{
    const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (e >= nentry) return;
    const double iw = 1.0 / w;
    double2 acc = {0, 0};
    for (int c = estart[e]; c < estart[e + 1]; ++c) {
        const int code = contrib[c];
        const int i = code / 9, s = (code / 3) % 3, u = code % 3;
        acc = cadd(acc, slot_value(g, P[i], Q[i], s, u, M + 7 * (size_t)i, w, iw));
    }
    TZ *z = Z + (size_t)erow[e] * ld + ecol[e];
    if constexpr (sizeof(TZ) == 16) {
        double2 v = *(double2 *)z;
        *(double2 *)z = cadd(v, acc);
    } else {
        float2 v = *(float2 *)z;
        *(float2 *)z = make_float2(v.x + (float)acc.x, v.y + (float)acc.y);
    }
}

// the 9 COO triplets of each pair (mom25d_core.cpp:477-506, mode 2)
__global__ void k_near_coo(DMesh g, const int *P, const int *Q, const double2 *M, long n, double w, int *ri, int *ci,
                           double2 *vv)
{
    const long idx = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (idx >= 9 * n) return;
    const long i = idx / 9;
    const int s = (int)((idx / 3) % 3), u = (int)(idx % 3);
    const int p = P[i], q = Q[i];
    const int em_ = g.te[3 * p + s], en = g.te[3 * q + u];
    if (em_ < 0 || en < 0) {
        ri[idx] = -1; ci[idx] = 0; vv[idx] = make_double2(0, 0);
        return;
    }
    ri[idx] = em_; ci[idx] = en;
    vv[idx] = slot_value(g, p, q, s, u, M + 7 * (size_t)i, w, 1.0 / w);
}

// ---- near pairs: brute force, one workgroup per triangle p, q in order ------------------------------------
__device__ inline bool is_near(const double *c, const double *sz, const double *zz, int p, int q, double fac)
{
    const double dx = c[2 * p] - c[2 * q], dy = c[2 * p + 1] - c[2 * q + 1], dz = zz[p] - zz[q];
    const double R = fac * fmax(sz[p], sz[q]);
    return dx * dx + dy * dy + dz * dz < R * R;
}

__global__ __launch_bounds__(256) void k_near_count(const double *c, const double *sz, const double *zz, int Nt,
                                                    double fac, long long *counts)
{
    const int p = blockIdx.x;
    __shared__ int part[256];
    int k = 0;
    for (int q = threadIdx.x; q < Nt; q += 256) k += is_near(c, sz, zz, p, q, fac);
    part[threadIdx.x] = k;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) part[threadIdx.x] += part[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) counts[p] = part[0];
}

__global__ __launch_bounds__(256) void k_near_write(const double *c, const double *sz, const double *zz, int Nt,
                                                    double fac, const long long *offs, int *P, int *Q)
{
    const int p = blockIdx.x;
    __shared__ int scan[256];
    __shared__ long long base;
    if (threadIdx.x == 0) base = offs[p];
    __syncthreads();
    for (int q0 = 0; q0 < Nt; q0 += 256) {
        const int q = q0 + threadIdx.x;
        const int f = (q < Nt) && is_near(c, sz, zz, p, q, fac);
        scan[threadIdx.x] = f;
        __syncthreads();
        for (int s = 1; s < 256; s <<= 1) {                 // inclusive Hillis-Steele scan
            const int v = (int)threadIdx.x >= s ? scan[threadIdx.x - s] : 0;
            __syncthreads();
            scan[threadIdx.x] += v;
            __syncthreads();
        }
        if (f) {
            const long long at = base + scan[threadIdx.x] - 1;
            P[at] = p; Q[at] = q;
        }
        __syncthreads();
        if (threadIdx.x == 255) base += scan[255];
        __syncthreads();
    }
}

// ---- fan columns and radial sums ---------------------------------------------------------------------------
__global__ void k_fan_q(DMesh g, DTab T, const int *F, int nf, double2 *o)
{
    const long idx = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (idx >= (long)g.Nt * nf) return;
    const int t = (int)(idx / nf), j = (int)(idx % nf);
    const int f = F[j];
    double2 ga, gq;
    tab_kern(T, g.lt[t], g.lt[f], cdist(g.cent, t, f), ga, gq);
    o[idx] = cscale(gq, g.area[t] * g.area[f]);
}

__global__ void k_radial(const double *x, const double *y, const double *W, long nt, long nq, const double *ax,
                         const double *ay, long nv, const double2 *d, long n, double dr, double2 *o)
{
    const long idx = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (idx >= nt * nv) return;
    const long t = idx / nv, v = idx % nv;
    const double top = (double)n - 1.000001;
    double2 acc = {0, 0};
    for (long q = 0; q < nq; ++q) {
        const double rx = x[t * nq + q] - ax[v], ry = y[t * nq + q] - ay[v];
        double u = hypot(rx, ry) / dr;
        if (!(u <= top)) u = top;
        const long i = (long)u;
        const double f = u - (double)i;
        const double2 a = d[i], b = d[i + 1];
        const double wt = W[t * nq + q];
        acc = cadd(acc, cscale(make_double2(a.x * (1.0 - f) + b.x * f, a.y * (1.0 - f) + b.y * f), wt));
    }
    o[idx] = acc;
}

// ---- Bessel functions of complex argument (power series / Hankel's asymptotic expansion, Abramowitz &
// Stegun 9.1.10 and 9.2.5; the reference's bessel_jn_complex1, mom25d_core.cpp:1515-1549) ---------------------
__device__ inline double c_abs(double2 z) { return hypot(z.x, z.y); }
__device__ inline double2 c_sqrt(double2 z)
{
    const double r = c_abs(z);
    if (r == 0.0) return make_double2(0.0, z.y);
    if (z.x >= 0) {
        const double t = sqrt(0.5 * (r + z.x));
        return make_double2(t, z.y / (2 * t));
    }
    const double t = sqrt(0.5 * (r - z.x));
    return make_double2(fabs(z.y) / (2 * t), copysign(t, z.y));
}
__device__ inline double2 c_cos(double2 z) { return make_double2(cos(z.x) * cosh(z.y), -sin(z.x) * sinh(z.y)); }
__device__ inline double2 c_sin(double2 z) { return make_double2(sin(z.x) * cosh(z.y), cos(z.x) * sinh(z.y)); }

__device__ double2 bessel_jn_c(int n, double2 z)
{
    const double PI = 3.14159265358979323846;
    const double az = c_abs(z);
    if (az <= 14.0) {
        const double2 h = cscale(z, 0.5);
        const double2 mh2 = cscale(cmul(h, h), -1.0);
        double2 term = n == 0 ? make_double2(1.0, 0.0) : n == 1 ? h : cscale(cmul(h, h), 0.5);
        double2 sum = term;
        double big = c_abs(term);
        for (int k = 1; k < 300; ++k) {
            term = cmul(term, cscale(mh2, 1.0 / ((double)k * (double)(k + n))));
            sum = cadd(sum, term);
            const double at = c_abs(term);
            big = fmax(big, at);
            if (k > az && at <= 1e-18 * big) break;
        }
        return sum;
    }
    const double mu = 4.0 * n * n;
    const double2 iz = cdiv(make_double2(1.0, 0.0), z);
    const double2 chi = make_double2(z.x - (0.5 * n + 0.25) * PI, z.y);
    double2 Pp = {1.0, 0.0}, Qq = {0.0, 0.0}, t = {1.0, 0.0};
    double prev = 1.0;
    for (int k = 1; k < 80; ++k) {
        const double m = 2.0 * k - 1.0;
        const double2 nt = cmul(cscale(t, (mu - m * m) / (8.0 * k)), iz);
        const double at = c_abs(nt);
        if (at >= prev) break;
        t = nt; prev = at;
        const double sg = ((k / 2) & 1) ? -1.0 : 1.0;
        if (k & 1) Qq = cadd(Qq, cscale(t, sg)); else Pp = cadd(Pp, cscale(t, sg));
        if (at < 1e-17) break;
    }
    const double2 pre = c_sqrt(cdiv(make_double2(2.0, 0.0), cscale(z, PI)));
    return cmul(pre, csub(cmul(Pp, c_cos(chi)), cmul(Qq, c_sin(chi))));
}

__global__ void k_bessel(int n, const double2 *z, long total, double2 *o)
{
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < total) o[i] = bessel_jn_c(n, z[i]);
}

// out[s, i] = sum_k J0(rho_i kr_k) W[s, k]: one workgroup per rho; the real nodes and the lifted ones summed
// apart and added at the end, as the reference adds its two parts (via.py:97-101). Several sets of distances, each with
// rows of its own, go in one launch (a set of 200 or 260 distances alone leaves the chip two thirds empty: a launch of one
// took 53 us, three of them in one launch take 64).
constexpr int HS = 4;
struct HankelSets {
    int n;
    double scale;                               // the sums are divided by it
    m25x_hankel_set set[M25X_HANKEL_SETS];
};
__global__ __launch_bounds__(256) void k_hankel(HankelSets hs, const double *rho, const double2 *kr, int nk,
                                                const double2 *W, double2 *out)
{
    int q = 0;
    while (q + 1 < hs.n && (int)blockIdx.x >= hs.set[q + 1].first) ++q;
    const int i = (int)blockIdx.x - hs.set[q].first, nr = hs.set[q].count, ns = hs.set[q].rows;
    const double r = rho[blockIdx.x];
    W += (size_t)hs.set[q].row * nk;
    out += hs.set[q].out;
    __shared__ double2 red[2][HS][256];
    for (int s0 = 0; s0 < ns; s0 += HS) {
        double2 aR[HS], aC[HS];
#pragma unroll
        for (int s = 0; s < HS; ++s) { aR[s] = make_double2(0, 0); aC[s] = make_double2(0, 0); }
        for (int k = threadIdx.x; k < nk; k += 256) {
            const double2 z = kr[k];
            if (fabs(z.y) < 1e-300) {
                const double j = j0(r * z.x);
#pragma unroll
                for (int s = 0; s < HS; ++s)
                    if (s0 + s < ns) aR[s] = cadd(aR[s], cscale(W[(size_t)(s0 + s) * nk + k], j));
            } else {
                const double2 J = bessel_jn_c(0, make_double2(r * z.x, r * z.y));
#pragma unroll
                for (int s = 0; s < HS; ++s)
                    if (s0 + s < ns) aC[s] = cadd(aC[s], cmul(J, W[(size_t)(s0 + s) * nk + k]));
            }
        }
#pragma unroll
        for (int s = 0; s < HS; ++s) { red[0][s][threadIdx.x] = aR[s]; red[1][s][threadIdx.x] = aC[s]; }
        __syncthreads();
        for (int st = 128; st > 0; st >>= 1) {
            if ((int)threadIdx.x < st) {
#pragma unroll
                for (int s = 0; s < HS; ++s) {
                    red[0][s][threadIdx.x] = cadd(red[0][s][threadIdx.x], red[0][s][threadIdx.x + st]);
                    red[1][s][threadIdx.x] = cadd(red[1][s][threadIdx.x], red[1][s][threadIdx.x + st]);
                }
            }
            __syncthreads();
        }
        if (threadIdx.x < HS && s0 + (int)threadIdx.x < ns) {
            const double2 v = cadd(red[0][threadIdx.x][0], red[1][threadIdx.x][0]);
            out[(size_t)(s0 + threadIdx.x) * nr + i] = make_double2(v.x / hs.scale, v.y / hs.scale);
        }
        __syncthreads();
    }
}

// ---- tables on the uniform grid ------------------------------------------------------------------------------
// out[row][i] = sum_j S[i][j] y[row][j], S given transposed (nc x nfine) so that a wave's loads of it are whole lines;
// a lane a fine point, RS rows a thread, a quarter of the nodes a wave, whose loads are asked for many at a time; the
// rows' coarse values in LDS. pairs: rows 2 t and 2 t + 1 side by side per point (the tables' A and Q). Reading S, 8192
// x 260 doubles, bounds it: 14 us with S in the caches, 28 without (a point finds it there no more); the library's two
// real products and the copies into this layout took 60 us more.
constexpr int RS = 4, RP = 64, RG = 4;       // rows a thread, points and node groups of a workgroup
constexpr int RN = 512, RU = 22;             // coarse nodes in LDS at a time; loads of S in flight a thread
__global__ __launch_bounds__(RP * RG) void k_resample(const double *St, int nc, int nfine, const double2 *y, int rows,
                                                      int pairs, double2 *out)
{
    __shared__ double2 yl[RN * RS];             // [node][row]; the groups' sums at the end
    const int lane = threadIdx.x % RP, g = threadIdx.x / RP;
    const int i = blockIdx.x * RP + lane, r0 = blockIdx.y * RS, ic = i < nfine ? i : nfine - 1;
    double2 acc[RS];
#pragma unroll
    for (int r = 0; r < RS; ++r) acc[r] = make_double2(0.0, 0.0);
    for (int j0 = 0; j0 < nc; j0 += RN) {
        const int nj = nc - j0 < RN ? nc - j0 : RN, per = (nj + RG - 1) / RG;
        if (j0) __syncthreads();
        for (int e = threadIdx.x; e < nj * RS; e += RP * RG) {
            const int r = r0 + e / nj, j = e % nj;
            yl[j * RS + e / nj] = y[(size_t)(r < rows ? r : rows - 1) * nc + j0 + j];
        }
        __syncthreads();
        const int ja = g * per, jb = ja + per < nj ? ja + per : nj;
        for (int j = ja; j < jb; j += RU) {
            double w[RU];                       // the group's next entries of S, all asked for first
#pragma unroll
            for (int u = 0; u < RU; ++u) w[u] = St[(size_t)(j0 + (j + u < jb ? j + u : jb - 1)) * nfine + ic];
#pragma unroll
            for (int u = 0; u < RU; ++u) {
                if (j + u >= jb) break;
#pragma unroll
                for (int r = 0; r < RS; ++r) acc[r] = cadd(acc[r], cscale(yl[(j + u) * RS + r], w[u]));
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS; ++r) yl[(g * RS + r) * RP + lane] = acc[r];
    __syncthreads();
    const int row = r0 + g;                     // group g adds up row g
    if (i >= nfine || row >= rows) return;
    double2 v = yl[g * RP + lane];
#pragma unroll
    for (int h = 1; h < RG; ++h) v = cadd(v, yl[(h * RS + g) * RP + lane]);
    out[pairs ? ((size_t)(row >> 1) * nfine + i) * 2 + (row & 1) : (size_t)row * nfine + i] = v;
}
static_assert(RG == RS && RG * RS * RP <= RN * RS, "a group per row, and room for the sums");

// ---- via blocks ----------------------------------------------------------------------------------------------
// QF += the near pairs' correction of the fan moments
__global__ void k_fan_add(m25x_via v, const double2 *qc, double2 *QF)
{
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= v.nfan) return;
    double2 *o = QF + (size_t)v.fan_row[i] * v.nF + v.fan_col[i];
    *o = cadd(*o, qc[v.fan_sel[i]]);
}

// X[t, n] = the potential of chain n on triangle t: its end charges' through the fan moments, and its smooth kernel
// D(layer of t, span of n) over the triangle's six points
__global__ void k_via_tri(m25x_via v, const int *lt, const double *P6, const double *W6, double w, const double2 *QF,
                          const double2 *D, double dr, double2 *X)
{
    const long idx = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (idx >= (long)v.Nt * v.Nv) return;
    const int t = (int)(idx / v.Nv), c = (int)(idx % v.Nv);
    double2 pot = {0, 0}, acc = {0, 0};
    for (int j = 0; j < v.nF; ++j) pot = cadd(pot, cscale(QF[(size_t)t * v.nF + j], v.dF[(size_t)j * v.Nv + c]));
    const double2 *d = D + (size_t)(v.span[c] * v.nlayer + lt[t]) * v.nfine;
    const double top = (double)v.nfine - 1.000001;
    for (int q = 0; q < 6; ++q) {
        const double rx = P6[(size_t)t * 12 + 2 * q] - v.vx[c], ry = P6[(size_t)t * 12 + 2 * q + 1] - v.vy[c];
        double u = hypot(rx, ry) / dr;
        if (!(u <= top)) u = top;
        const long i = (long)u;
        const double f = u - (double)i;
        const double2 a = d[i], b = d[i + 1];
        acc = cadd(acc, cscale(make_double2(a.x * (1.0 - f) + b.x * f, a.y * (1.0 - f) + b.y * f), W6[(size_t)t * 6 + q]));
    }
    X[idx] = make_double2(acc.x + pot.y / w, acc.y - pot.x / w);            // pot / (j w)
}

// B[e, n] = wp X[T+] + wm X[T-]
__global__ void k_via_div(m25x_via v, const double2 *X, double2 *B)
{
    const long idx = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (idx >= (long)v.Ne * v.Nv) return;
    const int e = (int)(idx / v.Nv), c = (int)(idx % v.Nv);
    B[idx] = cadd(cscale(X[(size_t)v.tp[e] * v.Nv + c], v.wp[e]), cscale(X[(size_t)v.tm[e] * v.Nv + c], v.wm[e]));
}

// C[m, n] = C0[m, n] + R[pair(m, n)] + the end charges' part: a wave an entry, a lane a fan triangle (in turns)
__global__ __launch_bounds__(64) void k_via_c(m25x_via v, double w, const double2 *QF, const double2 *R, const double2 *C0,
                                              double2 *Cv)
{
    const int m = blockIdx.x / v.Nv, c = blockIdx.x % v.Nv;
    double2 acc = {0, 0};
    for (int i = threadIdx.x; i < v.nF; i += 64) {
        const double dm = v.dF[(size_t)i * v.Nv + m];
        if (dm == 0.0) continue;
        double2 pot = {0, 0};
        const double2 *q = QF + (size_t)v.F[i] * v.nF;
        for (int j = 0; j < v.nF; ++j) pot = cadd(pot, cscale(q[j], v.dF[(size_t)j * v.Nv + c]));
        acc = cadd(acc, cscale(pot, dm));
    }
    __shared__ double2 red[64];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int st = 32; st > 0; st >>= 1) {
        if ((int)threadIdx.x < st) red[threadIdx.x] = cadd(red[threadIdx.x], red[threadIdx.x + st]);
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const int p = v.pair[blockIdx.x];
        double2 o = C0[blockIdx.x];
        if (p >= 0) o = cadd(o, R[p]);
        Cv[blockIdx.x] = make_double2(o.x + red[0].y / w, o.y - red[0].x / w);
    }
}

// ---- equilibration -------------------------------------------------------------------------------------------
// Z <- (Z d_i) d_j in place (fast.py:300-303: rows, then columns) and its complex64 copy
__global__ void k_scale(double2 *Z, long n, long ld, const double *d, float2 *Z64, long ld64)
{
    const long j = blockIdx.x * (long)blockDim.x + threadIdx.x;
    const long i = blockIdx.y;
    if (j >= n) return;
    const double di = d[i], dj = d[j];
    double2 z = Z[i * ld + j];
    z.x = (z.x * di) * dj; z.y = (z.y * di) * dj;
    Z[i * ld + j] = z;
    if (Z64) Z64[i * ld64 + j] = make_float2((float)z.x, (float)z.y);
}

__global__ void k_diag_scales(const double2 *Z, long n, long ld, double *d)
{
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double2 z = Z[i * ld + i];
    d[i] = 1.0 / sqrt(hypot(z.x, z.y) + 1e-300);
}

inline unsigned blocks(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// ---- the far product without Z (matvec_far, matvec_far_multi) ---------------------------------------------
// Three passes: the sources of each triangle aggregated (per column c: s0 = sum a x_e, s1 = sum a x_e (c_t - v_e)
// over its edges, a = alpha_e area_t), one kernel evaluation per triangle pair for all k columns (each workgroup
// a block of observation triangles against one slice of the sources, partial sums kept per slice), and each
// edge's two halves from the slices summed in slice order. Deterministic: no atomics, fixed orders.
constexpr int MV_P = 128;      // observation triangles a workgroup, one a thread
constexpr int MV_Q = 64;       // source triangles staged in LDS a step
constexpr int MV_KMAX = 8;     // columns a call

// slices of the sources: enough workgroups to fill the chip (about 1024), each slice a multiple of MV_Q
inline void mv_slices(int Nt, int &nslice, int &qper)
{
    const int pblocks = (Nt + MV_P - 1) / MV_P;
    int want = (1024 + pblocks - 1) / pblocks;
    want = want < 1 ? 1 : (want > 64 ? 64 : want);
    qper = (Nt + want - 1) / want;
    qper = (qper + MV_Q - 1) / MV_Q * MV_Q;
    if (qper < MV_Q) qper = MV_Q;
    nslice = (Nt + qper - 1) / qper;
    if (nslice < 1) nslice = 1;
}

// S[(t k + c) 3 + {0, 1, 2}] = (s0, s1x, s1y); the triangle's edges in increasing index (the reference's edge loop
// adds them in that order); act[t]: some edge has t as a half
__global__ void k_mv_sources(DMesh g, const double2 *X, long ldx, int k, double2 *S, int *act)
{
    const long idx = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (idx >= (long)g.Nt * k) return;
    const int t = (int)(idx / k), c = (int)(idx % k);
    int e3[3], n = 0;
    for (int i = 0; i < 3; ++i) {
        const int e = g.te[3 * t + i];
        if (e >= 0) e3[n++] = e;
    }
    for (int i = 1; i < n; ++i)
        for (int j = i; j > 0 && e3[j - 1] > e3[j]; --j) {
            const int x = e3[j]; e3[j] = e3[j - 1]; e3[j - 1] = x;
        }
    double2 s0 = {0, 0}, sx = {0, 0}, sy = {0, 0};
    const double cx = g.cent[2 * t], cy = g.cent[2 * t + 1];
    for (int j = 0; j < n; ++j) {
        const int e = e3[j];
        const bool plus = g.ep[e] == t;
        const double f = (plus ? g.ap[e] : g.am[e]) * g.area[t];
        const double *v = (plus ? g.vp : g.vm) + 2 * (size_t)e;
        const double2 xe = X[(size_t)e * ldx + c];
        const double2 a = make_double2(f * xe.x, f * xe.y);
        s0 = cadd(s0, a);
        sx = cadd(sx, cscale(a, cx - v[0]));
        sy = cadd(sy, cscale(a, cy - v[1]));
    }
    S[3 * idx] = s0; S[3 * idx + 1] = sx; S[3 * idx + 2] = sy;
    if (c == 0) act[t] = n > 0;
}

// part[((slice Nt + p) k + c) 3 + {0, 1, 2}] = sum over the slice's active q of (G_A s1x, G_A s1y, G_q s0)
template <int KM>
__global__ __launch_bounds__(MV_P) void k_mv_pairs(DMesh g, DTab T, const double2 *S, const int *act, int k,
                                                   int qper, double2 *part)
{
    __shared__ double2 sS[MV_Q][3 * KM];
    __shared__ double2 sc[MV_Q];
    __shared__ int sl[MV_Q];
    const int p = blockIdx.x * MV_P + threadIdx.x;
    const int q0 = blockIdx.y * qper, q1 = min(g.Nt, q0 + qper);
    const bool live = p < g.Nt;
    const int lp = live ? g.lt[p] : 0;
    const double px = live ? g.cent[2 * p] : 0.0, py = live ? g.cent[2 * p + 1] : 0.0;
    double2 ax[KM], ay[KM], aq[KM];
#pragma unroll
    for (int c = 0; c < KM; ++c) ax[c] = ay[c] = aq[c] = make_double2(0, 0);
    for (int qb = q0; qb < q1; qb += MV_Q) {
        const int nq = min(MV_Q, q1 - qb);
        for (int i = threadIdx.x; i < nq * 3 * k; i += MV_P) {
            const int j = i / (3 * k), r = i % (3 * k);
            sS[j][r] = S[(size_t)(qb + j) * 3 * k + r];
        }
        for (int j = threadIdx.x; j < nq; j += MV_P) {
            sc[j] = make_double2(g.cent[2 * (qb + j)], g.cent[2 * (qb + j) + 1]);
            sl[j] = act[qb + j] ? g.lt[qb + j] : -1;
        }
        __syncthreads();
        if (live) {
            for (int j = 0; j < nq; ++j) {
                const int lq = sl[j];
                if (lq < 0) continue;
                const double dx = px - sc[j].x, dy = py - sc[j].y;
                double2 ga, gq;
                tab_kern(T, lp, lq, sqrt(dx * dx + dy * dy), ga, gq);
#pragma unroll
                for (int c = 0; c < KM; ++c) {
                    if (c < k) {
                        ax[c] = cadd(ax[c], cmul(ga, sS[j][3 * c + 1]));
                        ay[c] = cadd(ay[c], cmul(ga, sS[j][3 * c + 2]));
                        aq[c] = cadd(aq[c], cmul(gq, sS[j][3 * c]));
                    }
                }
            }
        }
        __syncthreads();
    }
    if (!live) return;
    double2 *o = part + ((size_t)blockIdx.y * g.Nt + p) * k * 3;
#pragma unroll
    for (int c = 0; c < KM; ++c)
        if (c < k) { o[3 * c] = ax[c]; o[3 * c + 1] = ay[c]; o[3 * c + 2] = aq[c]; }
}

// The slices of part summed in slice order, into slice 0: one thread a value. (As a part of the edges' pass, whose
// threads each walked six values' slices, the sums took 27 us at 2560 triangles and 4 columns; 11 us and 3 us apart.)
__global__ void k_mv_slices(double2 *part, int nslice, long nv)
{
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= nv) return;
    double2 v = part[i];
    for (int sl = 1; sl < nslice; ++sl) v = cadd(v, part[sl * nv + i]);
    part[i] = v;
}

// Y[e, c] = sum over the halves (t, alpha, v) of alpha area_t [jw ((c_t - v) . vA_t) + 4 wQ_t / (jw)]
// (mom25d_core.cpp:300-311)
__global__ void k_mv_out(DMesh g, const double2 *part, int k, double w, double2 *Y, long ldy)
{
    const long idx = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (idx >= (long)g.Ne * k) return;
    const int e = (int)(idx / k), c = (int)(idx % k);
    const double iw = 1.0 / w;
    double2 y = {0, 0};
    for (int h = 0; h < 2; ++h) {
        const int t = h ? g.em[e] : g.ep[e];
        const double f = (h ? g.am[e] : g.ap[e]) * g.area[t];
        const double *v = (h ? g.vm : g.vp) + 2 * (size_t)e;
        const double dx = g.cent[2 * t] - v[0], dy = g.cent[2 * t + 1] - v[1];
        const double2 *o = part + ((size_t)t * k + c) * 3;
        const double2 vx = o[0], vy = o[1], wq = o[2];
        const double2 u = make_double2(dx * vx.x + dy * vy.x, dx * vx.y + dy * vy.y);
        // jw u + 4 wQ / (jw)
        const double2 z = make_double2(-w * u.y + 4.0 * wq.y * iw, w * u.x - 4.0 * wq.x * iw);
        y = cadd(y, cscale(z, f));
    }
    Y[(size_t)e * ldy + c] = y;
}

// ---- the near correction as a sparse operator ------------------------------------------------------------
// vals[e] = the correction of near entry e (its contributions in their fixed order, as k_near_scatter adds them)
__global__ __launch_bounds__(256) void k_near_values(DMesh g, const int *P, const int *Q, const double2 *M,
                                                     long nentry, const int *estart, const int *contrib, double w,
                                                     double2 *vals)
{
    const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (e >= nentry) return;
    const double iw = 1.0 / w;
    double2 acc = {0, 0};
    for (int c = estart[e]; c < estart[e + 1]; ++c) {
        const int code = contrib[c];
        const int i = code / 9, s = (code / 3) % 3, u = code % 3;
        acc = cadd(acc, slot_value(g, P[i], Q[i], s, u, M + 7 * (size_t)i, w, iw));
    }
    vals[e] = acc;
}

// Y[r, c] (+)= sum over the entries of row r of vals[e] X[col[e], c]: a wave a row, its lanes over the row's entries (so
// vals and col are read in order), all KM columns at once, the lanes' sums added by a fixed exchange. A thread a (row,
// column) walked 300 entries one after the other: 109 us at 3512 rows and 4 columns, 12 us so.
template <int KM>
__global__ __launch_bounds__(256) void k_csr_matvec(const int *rowptr, const int *col, const double2 *vals, long nrow,
                                                    const double2 *X, int k, long ldx, double2 *Y, long ldy, int add)
{
    const long r = blockIdx.x * 4L + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (r >= nrow) return;
    double sx[KM], sy[KM];
#pragma unroll
    for (int c = 0; c < KM; ++c) sx[c] = sy[c] = 0.0;
    const int e1 = rowptr[r + 1];
    for (int e = rowptr[r] + lane; e < e1; e += 64) {
        const double2 a = vals[e];
        const double2 *x = X + (size_t)col[e] * ldx;
#pragma unroll
        for (int c = 0; c < KM; ++c)
            if (c < k) {
                const double2 p = cmul(a, x[c]);
                sx[c] += p.x; sy[c] += p.y;
            }
    }
#pragma unroll
    for (int c = 0; c < KM; ++c) {
        for (int o = 32; o > 0; o >>= 1) { sx[c] += __shfl_xor(sx[c], o); sy[c] += __shfl_xor(sy[c], o); }
        if (lane == c && c < k) {
            double2 *y = Y + r * ldy + c;
            const double2 s = make_double2(sx[c], sy[c]);
            *y = add ? cadd(*y, s) : s;
        }
    }
}

// ---- the via rows and columns of the operator ---------------------------------------------------------------
// B (ne x nv) couples the edges and the via chains, C (nv x nv) the chains (row-major). The chains' rows
// Y[ne + v] = sum_e B[e, v] X[e] + sum_u C[v, u] X[ne + u] in two passes: a workgroup a chain and one of VB blocks of the
// edges, then the blocks in order with the edges' rows Y[e] += sum_v B[e, v] X[ne + v]. The product with B^T has few
// outputs and thousands of terms each: a library product gave it one workgroup (384 us at 3512 edges, 4 chains and 4
// columns; 8 us so).
constexpr int VB = 32;
template <int KM>
__global__ __launch_bounds__(256) void k_via_rows(const double2 *B, long ne, int nv, const double2 *X, int k, long ldx,
                                                  double2 *part)
{
    const int v = blockIdx.y, b = blockIdx.x, tid = threadIdx.x;
    const long rows = (ne + VB - 1) / VB, r0 = b * rows, r1 = min(ne, r0 + rows);
    double sx[KM], sy[KM];
#pragma unroll
    for (int c = 0; c < KM; ++c) sx[c] = sy[c] = 0.0;
    for (long e = r0 + tid; e < r1; e += 256) {
        const double2 a = B[e * nv + v];
#pragma unroll
        for (int c = 0; c < KM; ++c)
            if (c < k) {
                const double2 p = cmul(a, X[e * ldx + c]);
                sx[c] += p.x; sy[c] += p.y;
            }
    }
    __shared__ double2 red[4][KM];
#pragma unroll
    for (int c = 0; c < KM; ++c) {
        for (int o = 32; o > 0; o >>= 1) { sx[c] += __shfl_xor(sx[c], o); sy[c] += __shfl_xor(sy[c], o); }
        if ((tid & 63) == 0) red[tid >> 6][c] = make_double2(sx[c], sy[c]);
    }
    __syncthreads();
    if (tid < k) part[((size_t)v * VB + b) * k + tid] = cadd(cadd(red[0][tid], red[1][tid]), cadd(red[2][tid], red[3][tid]));
}

__global__ void k_via_out(const double2 *B, const double2 *C, long ne, int nv, const double2 *X, int k, long ldx,
                          const double2 *part, double2 *Y, long ldy)
{
    const long idx = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (idx >= (ne + nv) * k) return;
    const long r = idx / k;
    const int c = (int)(idx % k);
    const double2 *a = r < ne ? B + r * nv : C + (r - ne) * nv;
    double2 s = {0, 0};
    for (int u = 0; u < nv; ++u) s = cadd(s, cmul(a[u], X[(ne + u) * ldx + c]));
    if (r < ne) s = cadd(Y[r * ldy + c], s);
    else
        for (int b = 0; b < VB; ++b) s = cadd(s, part[((size_t)(r - ne) * VB + b) * k + c]);
    Y[r * ldy + c] = s;
}

}  // namespace

extern "C" {

int m25x_fill_far(void *Z, int zdtype, long ld, const m25x_mesh *g, const m25x_tables *tb, double w, void *stream)
{
    if (!Z || !g || !tb || ld < g->Ne || !(w > 0)) return fail(M25X_EINVAL, "fill_far: bad arguments");
    if (g->Ne == 0) return M25X_OK;
    const int nt = (g->Ne + FT - 1) / FT;
    dim3 grid(nt, nt);
    hipStream_t s = (hipStream_t)stream;
    TimedLaunch tl(s, M25X_K_FILL_FAR, zdtype, (zdtype == M25X_C128 ? 16.0 : 8.0) * g->Ne * (double)g->Ne, 0.0);
    if (zdtype == M25X_C128)
        hipLaunchKernelGGL(k_fill_far<double2>, grid, dim3(FTH), 0, s, (double2 *)Z, ld, dmesh(g), dtab(tb), w);
    else if (zdtype == M25X_C64)
        hipLaunchKernelGGL(k_fill_far<float2>, grid, dim3(FTH), 0, s, (float2 *)Z, ld, dmesh(g), dtab(tb), w);
    else
        return fail(M25X_EINVAL, "fill_far: zdtype %d", zdtype);
    return check_launch("fill_far");
}

int m25x_far_block(const int *rows, int nr, const int *cols, int nc, const m25x_mesh *g, const m25x_tables *tb,
                   double w, double *out, void *stream)
{
    if (nr < 0 || nc < 0 || !g || !tb) return fail(M25X_EINVAL, "far_block: bad arguments");
    if ((long)nr * nc == 0) return M25X_OK;
    hipLaunchKernelGGL(k_far_block, dim3(blocks((long)nr * nc, 256)), dim3(256), 0, (hipStream_t)stream, rows, nr,
                       cols, nc, dmesh(g), dtab(tb), w, (double2 *)out);
    return check_launch("far_block");
}

int m25x_near_moments(const m25x_mesh *g, const m25x_tables *tb, const m25x_quad *q, const int *P, const int *Q,
                      long n, double w, double *stat, int stat_ready, double *M, double *qcorr, void *stream)
{
    if (!g || !tb || !q || n < 0 || !M) return fail(M25X_EINVAL, "near_moments: bad arguments");
    if (n == 0) return M25X_OK;
    DQuad d{q->nodes, q->tris, q->P3, q->W3, q->P6, q->W6};
    TimedLaunch tl((hipStream_t)stream, M25X_K_NEAR_MOMENTS, M25X_C128, 7.0 * 16 * n, 0.0);
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid(blocks(n, 256));
    if (stat) {
        if (!stat_ready) hipLaunchKernelGGL(k_near_static, grid, dim3(256), 0, s, dmesh(g), dtab(tb), d, P, Q, n, stat);
        hipLaunchKernelGGL(k_near_moments<true>, grid, dim3(256), 0, s, dmesh(g), dtab(tb), d, P, Q, n, (const double *)stat,
                           (double2 *)M, (double2 *)qcorr);
    } else {
        hipLaunchKernelGGL(k_near_moments<false>, grid, dim3(256), 0, s, dmesh(g), dtab(tb), d, P, Q, n,
                           (const double *)nullptr, (double2 *)M, (double2 *)qcorr);
    }
    return check_launch("near_moments");
}

int m25x_near_scatter(void *Z, int zdtype, long ld, const m25x_mesh *g, const int *P, const int *Q, const double *M,
                      long nentry, const int *erow, const int *ecol, const int *estart, const int *contrib, double w,
                      void *stream)
{
    if (!Z || !g || nentry < 0) return fail(M25X_EINVAL, "near_scatter: bad arguments");
    if (nentry == 0) return M25X_OK;
    hipStream_t s = (hipStream_t)stream;
    TimedLaunch tl(s, M25X_K_NEAR_SCATTER, zdtype, (zdtype == M25X_C128 ? 32.0 : 16.0) * nentry, 0.0);
    if (zdtype == M25X_C128)
        hipLaunchKernelGGL(k_near_scatter<double2>, dim3(blocks(nentry, 256)), dim3(256), 0, s, (double2 *)Z, ld,
                           dmesh(g), P, Q, (const double2 *)M, nentry, erow, ecol, estart, contrib, w);
    else if (zdtype == M25X_C64)
        hipLaunchKernelGGL(k_near_scatter<float2>, dim3(blocks(nentry, 256)), dim3(256), 0, s, (float2 *)Z, ld,
                           dmesh(g), P, Q, (const double2 *)M, nentry, erow, ecol, estart, contrib, w);
    else
        return fail(M25X_EINVAL, "near_scatter: zdtype %d", zdtype);
    return check_launch("near_scatter");
}

size_t m25x_matvec_far_work_bytes(int Nt, int k)
{
    if (Nt <= 0 || k <= 0) return 256;
    int nslice, qper;
    mv_slices(Nt, nslice, qper);
    return sizeof(double2) * 3 * (size_t)Nt * k * (1 + (size_t)nslice) + sizeof(int) * (size_t)Nt + 256;
}

int m25x_matvec_far(const double *X, int k, long ldx, const m25x_mesh *g, const m25x_tables *tb, double w, double *Y,
                    long ldy, void *work, size_t work_bytes, void *stream)
{
    if (!X || !Y || !g || !tb || k < 1 || k > MV_KMAX || ldx < k || ldy < k || !(w > 0))
        return fail(M25X_EINVAL, "matvec_far: bad arguments (1 <= k <= %d, ldx, ldy >= k, w > 0)", MV_KMAX);
    if (g->Ne == 0) return M25X_OK;
    if (!work || work_bytes < m25x_matvec_far_work_bytes(g->Nt, k))
        return fail(M25X_EINVAL, "matvec_far: workspace of %zu bytes, %zu needed", work_bytes,
                    m25x_matvec_far_work_bytes(g->Nt, k));
    hipStream_t s = (hipStream_t)stream;
    int nslice, qper;
    mv_slices(g->Nt, nslice, qper);
    double2 *S = (double2 *)work, *part = S + 3 * (size_t)g->Nt * k;
    int *act = (int *)(part + 3 * (size_t)g->Nt * k * nslice);
    DMesh m = dmesh(g);
    hipLaunchKernelGGL(k_mv_sources, dim3(blocks((long)g->Nt * k, 256)), dim3(256), 0, s, m, (const double2 *)X, ldx,
                       k, S, act);
    if (int rc = check_launch("matvec_far")) return rc;
    const dim3 grid((g->Nt + MV_P - 1) / MV_P, nslice);
    if (k <= 1)
        hipLaunchKernelGGL(k_mv_pairs<1>, grid, dim3(MV_P), 0, s, m, dtab(tb), (const double2 *)S, (const int *)act,
                           k, qper, part);
    else if (k <= 4)
        hipLaunchKernelGGL(k_mv_pairs<4>, grid, dim3(MV_P), 0, s, m, dtab(tb), (const double2 *)S, (const int *)act,
                           k, qper, part);
    else
        hipLaunchKernelGGL(k_mv_pairs<MV_KMAX>, grid, dim3(MV_P), 0, s, m, dtab(tb), (const double2 *)S,
                           (const int *)act, k, qper, part);
    if (int rc = check_launch("matvec_far")) return rc;
    if (nslice > 1)
        hipLaunchKernelGGL(k_mv_slices, dim3(blocks(3L * g->Nt * k, 256)), dim3(256), 0, s, part, nslice, 3L * g->Nt * k);
    hipLaunchKernelGGL(k_mv_out, dim3(blocks((long)g->Ne * k, 256)), dim3(256), 0, s, m, (const double2 *)part, k, w,
                       (double2 *)Y, ldy);
    return check_launch("matvec_far");
}

int m25x_near_values(const m25x_mesh *g, const int *P, const int *Q, const double *M, long nentry, const int *estart,
                     const int *contrib, double w, double *vals, void *stream)
{
    if (!g || nentry < 0 || (nentry && (!P || !Q || !M || !estart || !contrib || !vals)))
        return fail(M25X_EINVAL, "near_values: bad arguments");
    if (nentry == 0) return M25X_OK;
    hipLaunchKernelGGL(k_near_values, dim3(blocks(nentry, 256)), dim3(256), 0, (hipStream_t)stream, dmesh(g), P, Q,
                       (const double2 *)M, nentry, estart, contrib, w, (double2 *)vals);
    return check_launch("near_values");
}

int m25x_csr_matvec(const int *rowptr, const int *col, const double *vals, long nrow, const double *X, int k, long ldx,
                    double *Y, long ldy, int add, void *stream)
{
    if (!rowptr || nrow < 0 || k < 1 || ldx < k || ldy < k || !X || !Y)
        return fail(M25X_EINVAL, "csr_matvec: bad arguments");
    if (nrow == 0) return M25X_OK;
    hipStream_t s = (hipStream_t)stream;
    const double2 *v = (const double2 *)vals, *x = (const double2 *)X;
    double2 *y = (double2 *)Y;
    for (int c0 = 0; c0 < k; c0 += MV_KMAX) {       // columns MV_KMAX at a time
        const int kc = k - c0 < MV_KMAX ? k - c0 : MV_KMAX;
        if (kc <= 1)
            hipLaunchKernelGGL(k_csr_matvec<1>, dim3(blocks(nrow, 4)), dim3(256), 0, s, rowptr, col, v, nrow, x + c0, kc,
                               ldx, y + c0, ldy, add);
        else if (kc <= 4)
            hipLaunchKernelGGL(k_csr_matvec<4>, dim3(blocks(nrow, 4)), dim3(256), 0, s, rowptr, col, v, nrow, x + c0, kc,
                               ldx, y + c0, ldy, add);
        else
            hipLaunchKernelGGL(k_csr_matvec<MV_KMAX>, dim3(blocks(nrow, 4)), dim3(256), 0, s, rowptr, col, v, nrow,
                               x + c0, kc, ldx, y + c0, ldy, add);
    }
    return check_launch("csr_matvec");
}

size_t m25x_via_matvec_work_bytes(int nv, int k)
{
    return nv > 0 && k > 0 ? sizeof(double2) * (size_t)VB * nv * (k < MV_KMAX ? k : MV_KMAX) : 16;
}

int m25x_via_matvec(const double *B, const double *C, long ne, int nv, const double *X, int k, long ldx, double *Y,
                    long ldy, void *work, size_t work_bytes, void *stream)
{
    if (ne < 0 || nv < 0 || k < 1 || ldx < k || ldy < k || !X || !Y || (nv && (!B || !C)))
        return fail(M25X_EINVAL, "via_matvec: bad arguments");
    if (nv == 0) return M25X_OK;
    if (!work || work_bytes < m25x_via_matvec_work_bytes(nv, k))
        return fail(M25X_EINVAL, "via_matvec: workspace of %zu bytes, %zu needed", work_bytes,
                    m25x_via_matvec_work_bytes(nv, k));
    hipStream_t s = (hipStream_t)stream;
    const double2 *b = (const double2 *)B, *c = (const double2 *)C, *x = (const double2 *)X;
    double2 *y = (double2 *)Y, *part = (double2 *)work;
    for (int c0 = 0; c0 < k; c0 += MV_KMAX) {
        const int kc = k - c0 < MV_KMAX ? k - c0 : MV_KMAX;
        if (kc <= 4)
            hipLaunchKernelGGL(k_via_rows<4>, dim3(VB, nv), dim3(256), 0, s, b, ne, nv, x + c0, kc, ldx, part);
        else
            hipLaunchKernelGGL(k_via_rows<MV_KMAX>, dim3(VB, nv), dim3(256), 0, s, b, ne, nv, x + c0, kc, ldx, part);
        hipLaunchKernelGGL(k_via_out, dim3(blocks((ne + nv) * kc, 256)), dim3(256), 0, s, b, c, ne, nv, x + c0, kc, ldx,
                           (const double2 *)part, y + c0, ldy);
    }
    return check_launch("via_matvec");
}

int m25x_near_coo(const m25x_mesh *g, const int *P, const int *Q, const double *M, long n, double w, int *ri, int *ci,
                  double *vv, void *stream)
{
    if (!g || n < 0) return fail(M25X_EINVAL, "near_coo: bad arguments");
    if (n == 0) return M25X_OK;
    hipLaunchKernelGGL(k_near_coo, dim3(blocks(9 * n, 256)), dim3(256), 0, (hipStream_t)stream, dmesh(g), P, Q,
                       (const double2 *)M, n, w, ri, ci, (double2 *)vv);
    return check_launch("near_coo");
}

int m25x_near_pairs(const double *cent, const double *size, const double *z, int Nt, double fac, long long *counts,
                    long *count, int *P, int *Q, void *stream)
{
    if (Nt < 0 || !counts || !count) return fail(M25X_EINVAL, "near_pairs: bad arguments");
    *count = 0;
    if (Nt == 0) return M25X_OK;
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(k_near_count, dim3(Nt), dim3(256), 0, s, cent, size, z, Nt, fac, counts);
    if (int rc = check_launch("near_pairs")) return rc;
    long long *h = (long long *)malloc(sizeof(long long) * ((size_t)Nt + 1));
    if (!h) return fail(M25X_ENOMEM, "near_pairs: host memory");
    hipError_t e = hipMemcpyAsync(h, counts, sizeof(long long) * Nt, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) { free(h); return fail(M25X_EHIP, "near_pairs: %s", hipGetErrorString(e)); }
    long long run = 0;
    for (int p = 0; p < Nt; ++p) { const long long c = h[p]; h[p] = run; run += c; }
    h[Nt] = run;
    *count = (long)run;
    if (P && Q && run > 0) {
        e = hipMemcpyAsync(counts, h, sizeof(long long) * ((size_t)Nt + 1), hipMemcpyHostToDevice, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        free(h);
        if (e != hipSuccess) return fail(M25X_EHIP, "near_pairs: %s", hipGetErrorString(e));
        hipLaunchKernelGGL(k_near_write, dim3(Nt), dim3(256), 0, s, cent, size, z, Nt, fac, counts, P, Q);
        return check_launch("near_pairs");
    }
    free(h);
    return M25X_OK;
}

int m25x_fan_q(const m25x_mesh *g, const m25x_tables *tb, const int *F, int nf, double *out, void *stream)
{
    if (!g || !tb || nf < 0) return fail(M25X_EINVAL, "fan_q: bad arguments");
    if ((long)g->Nt * nf == 0) return M25X_OK;
    hipLaunchKernelGGL(k_fan_q, dim3(blocks((long)g->Nt * nf, 256)), dim3(256), 0, (hipStream_t)stream, dmesh(g),
                       dtab(tb), F, nf, (double2 *)out);
    return check_launch("fan_q");
}

int m25x_radial_table_sum(const double *px, const double *py, const double *W, long nt, long nq, const double *vx,
                          const double *vy, long nv, const double *table, long n, double dr, double *out,
                          void *stream)
{
    if (n < 2 || !(dr > 0)) return fail(M25X_EINVAL, "radial_table_sum: a table of two points or more, dr > 0");
    if (nt < 0 || nq < 0 || nv < 0) return fail(M25X_EINVAL, "radial_table_sum: bad sizes");
    if (nt * nv == 0) return M25X_OK;
    hipLaunchKernelGGL(k_radial, dim3(blocks(nt * nv, 256)), dim3(256), 0, (hipStream_t)stream, px, py, W, nt, nq,
                       vx, vy, nv, (const double2 *)table, n, dr, (double2 *)out);
    return check_launch("radial_table_sum");
}

int m25x_hankel_sets(const double *rho, int nr, const m25x_hankel_set *sets, int nsets, double scale, const double *kr,
                     int nk, const double *W, int nrows, double *out, long nout, void *stream)
{
    if (nr < 0 || nk < 0 || nrows < 0 || nsets < 0 || nsets > M25X_HANKEL_SETS || (nsets && !sets))
        return fail(M25X_EINVAL, "hankel: bad sizes (at most %d sets)", M25X_HANKEL_SETS);
    HankelSets hs;
    hs.n = nsets;
    hs.scale = scale;
    int at = 0;
    for (int q = 0; q < nsets; ++q) {           // the sets cover the distances in order
        const m25x_hankel_set &t = hs.set[q] = sets[q];
        if (t.first != at || t.count < 0 || t.row < 0 || t.rows < 0 || t.row + t.rows > nrows || t.out < 0 ||
            t.out + (long)t.rows * t.count > nout)
            return fail(M25X_EINVAL, "hankel: set %d", q);
        at += t.count;
    }
    if (at != nr) return fail(M25X_EINVAL, "hankel: the sets cover %d of %d distances", at, nr);
    if (nr == 0) return M25X_OK;
    hipLaunchKernelGGL(k_hankel, dim3(nr), dim3(256), 0, (hipStream_t)stream, hs, rho, (const double2 *)kr, nk,
                       (const double2 *)W, (double2 *)out);
    return check_launch("hankel");
}

int m25x_hankel(const double *rho, int nr, const double *kr, int nk, const double *W, int ns, double *out,
                void *stream)
{
    if (nr < 0 || nk < 0 || ns < 0) return fail(M25X_EINVAL, "hankel: bad sizes");
    const m25x_hankel_set one = {0, nr, 0, ns, 0};
    return m25x_hankel_sets(rho, nr, &one, 1, 1.0, kr, nk, W, ns, out, (long)nr * ns, stream);
}

int m25x_resample(const double *St, int nc, int nfine, const double *y, int rows, int pairs, double *out, void *stream)
{
    if (nc < 1 || nfine < 0 || rows < 0 || (pairs && rows % 2))
        return fail(M25X_EINVAL, "resample: one node or more, an even number of rows for pairs");
    if (rows == 0 || nfine == 0) return M25X_OK;
    hipLaunchKernelGGL(k_resample, dim3(blocks(nfine, RP), blocks(rows, RS)), dim3(RP * RG), 0, (hipStream_t)stream,
                       St, nc, nfine, (const double2 *)y, rows, pairs, (double2 *)out);
    return check_launch("resample");
}

int m25x_via_blocks(const m25x_via *v, const m25x_mesh *g, const m25x_quad *q, double w, double *QF, const double *qc,
                    const double *D, double dr, const double *R, const double *C0, double *X, double *B, double *Cv,
                    void *stream)
{
    if (!v || !g || !q || v->Nv < 1 || v->Ne != g->Ne || v->Nt != g->Nt || v->nF < 0 || v->nfine < 2 || v->nfan < 0 ||
        !(dr > 0) || !(w > 0))
        return fail(M25X_EINVAL, "via_blocks: bad arguments");
    hipStream_t s = (hipStream_t)stream;
    if (v->nfan)
        hipLaunchKernelGGL(k_fan_add, dim3(blocks(v->nfan, 256)), dim3(256), 0, s, *v, (const double2 *)qc, (double2 *)QF);
    if (v->Nt)
        hipLaunchKernelGGL(k_via_tri, dim3(blocks((long)v->Nt * v->Nv, 256)), dim3(256), 0, s, *v, g->lt, q->P6, q->W6, w,
                           (const double2 *)QF, (const double2 *)D, dr, (double2 *)X);
    if (v->Ne)
        hipLaunchKernelGGL(k_via_div, dim3(blocks((long)v->Ne * v->Nv, 256)), dim3(256), 0, s, *v, (const double2 *)X,
                           (double2 *)B);
    hipLaunchKernelGGL(k_via_c, dim3(v->Nv * v->Nv), dim3(64), 0, s, *v, w, (const double2 *)QF, (const double2 *)R,
                       (const double2 *)C0, (double2 *)Cv);
    return check_launch("via_blocks");
}

int m25x_bessel_jn_complex(int n, const double *z, long total, double *out, void *stream)
{
    if (n < 0 || n > 2) return fail(M25X_EINVAL, "bessel_jn_complex: order 0, 1 or 2");
    if (total <= 0) return M25X_OK;
    hipLaunchKernelGGL(k_bessel, dim3(blocks(total, 256)), dim3(256), 0, (hipStream_t)stream, n,
                       (const double2 *)z, total, (double2 *)out);
    return check_launch("bessel_jn_complex");
}

int m25x_scale_c64(double *Z, long n, long ld, const double *d, float *Z64, long ld64, void *stream)
{
    if (!Z || !d || n < 0 || ld < n || (Z64 && ld64 < n)) return fail(M25X_EINVAL, "scale_c64: bad arguments");
    if (n == 0) return M25X_OK;
    hipLaunchKernelGGL(k_scale, dim3(blocks(n, 256), (unsigned)n), dim3(256), 0, (hipStream_t)stream, (double2 *)Z,
                       n, ld, d, (float2 *)Z64, ld64);
    return check_launch("scale_c64");
}

int m25x_diag_scales(const double *Z, long n, long ld, double *d, void *stream)
{
    if (!Z || !d || n < 0 || ld < n) return fail(M25X_EINVAL, "diag_scales: bad arguments");
    if (n == 0) return M25X_OK;
    hipLaunchKernelGGL(k_diag_scales, dim3(blocks(n, 256)), dim3(256), 0, (hipStream_t)stream, (const double2 *)Z,
                       n, ld, d);
    return check_launch("diag_scales");
}

}  // extern "C"
