// bt_hermite.hip -- the Hermite approximation on gfx950, in FP64.
//
// A Hermite cluster carries 8 planes per grid point (value, the three first,
// the three mixed second and the mixed third derivative terms, in the order
// 0, x, y, z, xy, yz, xz, xyz); the planes of node c sit at q[8*P*c + m*P + j]
// and its grid coordinates at x[P*c + j].  Per dimension, a point at
// displacement d from node k has the factors
//   A_k = dj_k / d^2 + w_k / d,   B_k = dj_k / d
// (dj = 1/4 at the two ends, 1 inside; w from the node's box), and plane m of
// the tensor grid point (k1,k2,k3) weighs the point by the product of one
// factor per dimension: A for a dimension that plane m does not
// differentiate, B for one it does.  A point on a node coordinate (|d| <
// DBL_MIN) takes A = [k == hit], B = 0 in that dimension and leaves that
// dimension out of its denominator (src/clusters/clusters.c:1224-1836,
// src/interaction_compute/interaction_compute_downpass.c:860-1109).
#include <hip/hip_runtime.h>

#include <cfloat>

#include "bt_exp.h"
#include "bt_kernels.h"
#include "bt_rsq.h"

namespace btk {
namespace {

constexpr int HTPB = 256;
constexpr int HCHUNK = 64;  // particles per LDS chunk of the upward pass
constexpr int HKC = 1, HKY = 2, HKR = 3, HKS = KERNEL_SIN_OVER_R;

__device__ __forceinline__ double herm_dj(int k, int n) { return (k == 0 || k == n) ? 0.25 : 1.0; }

// ---------------------------------------------------------------------
// Upward pass: block (part, slice) = particles [beg, end) of one node part
// against grid points slice*HTPB + tid; the 8 plane sums (8 more of w for
// subtraction) are stored to the part's row (partial rows are summed per
// node afterwards, in part order).
// ---------------------------------------------------------------------
template <int NL, bool SS>
__global__ __launch_bounds__(HTPB) void k_herm_anterp(HermAnterpArgs a)
{
    constexpr int n = NL - 1, P = NL * NL * NL;
    const int tid = threadIdx.x;
    const int part = blockIdx.x;
    const int node = a.part_node[part];
    const int beg = a.part_beg[part], end = a.part_end[part];
    const int j = blockIdx.y * HTPB + tid;
    const int jc = j < P ? j : 0;
    const int k1 = jc % NL, k2 = (jc / NL) % NL, k3 = jc / (NL * NL);

    __shared__ double Lnode[3][NL], Lw[3][NL];
    __shared__ double FA[3][NL][HCHUNK], FB[3][NL][HCHUNK];
    __shared__ double Lsum[3][HCHUNK], F1[HCHUNK], F2[HCHUNK];
    __shared__ int Lex[3][HCHUNK];
    if (tid < 3 * NL) {
        Lnode[tid / NL][tid % NL] = a.tab[(size_t)node * 3 * NL + tid];
        Lw[tid / NL][tid % NL] = a.wtab[(size_t)node * 3 * NL + tid];
    }

    double t[8], u[8];
#pragma unroll
    for (int m = 0; m < 8; m++) { t[m] = 0.0; u[m] = 0.0; }

    for (int base = beg; base < end; base += HCHUNK) {
        const int cnt = min(HCHUNK, end - base);
        __syncthreads();
        // factors of particle p in dimension d (thread d*HCHUNK + p)
        if (tid < 3 * HCHUNK) {
            const int d = tid / HCHUNK, p = tid % HCHUNK;
            if (p < cnt) {
                const double *pc = d == 0 ? a.px : (d == 1 ? a.py : a.pz);
                const double c = pc[base + p];
                int ex = -1;
                double sum = 0.0;
#pragma unroll
                for (int k = 0; k < NL; k++) {
                    const double dx = c - Lnode[d][k];
                    if (fabs(dx) < DBL_MIN) ex = k;
                    const double dj = herm_dj(k, n);
                    const double A = dj / (dx * dx) + Lw[d][k] / dx;
                    sum += A;
                    FA[d][k][p] = A;
                    FB[d][k][p] = dj / dx;
                }
                if (ex >= 0) {
#pragma unroll
                    for (int k = 0; k < NL; k++) { FA[d][k][p] = k == ex ? 1.0 : 0.0; FB[d][k][p] = 0.0; }
                }
                Lsum[d][p] = sum;
                Lex[d][p] = ex;
            } else {
#pragma unroll
                for (int k = 0; k < NL; k++) { FA[d][k][p] = 0.0; FB[d][k][p] = 0.0; }
            }
        }
        __syncthreads();
        // modified charges (clusters.c:1334-1370)
        if (tid < HCHUNK) {
            const int p = tid;
            double f1 = 0.0, f2 = 0.0;
            if (p < cnt) {
                double den = 1.0;
                if (Lex[0][p] == -1) den *= Lsum[0][p];
                if (Lex[1][p] == -1) den *= Lsum[1][p];
                if (Lex[2][p] == -1) den *= Lsum[2][p];
                const double q = a.pq[base + p];
                if constexpr (SS) {
                    const double w = a.pw[base + p];
                    f1 = q * w / den;
                    f2 = w / den;
                } else {
                    f1 = q / den;
                }
            }
            F1[p] = f1;
            F2[p] = f2;
        }
        __syncthreads();
        for (int p = 0; p < HCHUNK; p++) {
            const double ay = FA[1][k2][p], by = FB[1][k2][p], az = FA[2][k3][p], bz = FB[2][k3][p];
            const double yz00 = ay * az, yz10 = by * az, yz01 = ay * bz, yz11 = by * bz;
            const double xa = FA[0][k1][p] * F1[p], xb = FB[0][k1][p] * F1[p];
            t[0] = fma(xa, yz00, t[0]); t[1] = fma(xb, yz00, t[1]);
            t[2] = fma(xa, yz10, t[2]); t[3] = fma(xa, yz01, t[3]);
            t[4] = fma(xb, yz10, t[4]); t[5] = fma(xa, yz11, t[5]);
            t[6] = fma(xb, yz01, t[6]); t[7] = fma(xb, yz11, t[7]);
            if constexpr (SS) {
                const double wa = FA[0][k1][p] * F2[p], wb = FB[0][k1][p] * F2[p];
                u[0] = fma(wa, yz00, u[0]); u[1] = fma(wb, yz00, u[1]);
                u[2] = fma(wa, yz10, u[2]); u[3] = fma(wa, yz01, u[3]);
                u[4] = fma(wb, yz10, u[4]); u[5] = fma(wa, yz11, u[5]);
                u[6] = fma(wb, yz01, u[6]); u[7] = fma(wb, yz11, u[7]);
            }
        }
    }
    if (j < P) {
        double *q = a.Qp + (size_t)part * 8 * P;
#pragma unroll
        for (int m = 0; m < 8; m++) q[m * P + j] = t[m];
        if constexpr (SS) {
            double *w = a.Wp + (size_t)part * 8 * P;
#pragma unroll
            for (int m = 0; m < 8; m++) w[m * P + j] = u[m];
        }
    }
}

// ---------------------------------------------------------------------
// Particle-cluster far field: tile {key, first target, count} of up to
// HERM_PC_TILE targets against the 8-plane clusters of its key, added to the
// potential (coulomb_pc.c:66-135, yukawa_pc.c:61-140,
// regularized-coulomb_pc.c:67-139, coulomb_ss_pc.c:63-163,
// yukawa_ss_pc.c:61-167, regularized-coulomb_ss_pc.c:63-160).
//
// The launch issues FP64 instructions back to back, so the derivative
// expansion is written for few of them: the linear, bilinear and trilinear
// forms of the planes once each, then Horner in 1/r^2; and the points of a
// cluster's pencil (k2, k3) share dy, dz, dy^2 + dz^2 and dy dz.  Coulomb: 21
// instructions per pair and 5 per pencil, where the reference's expressions
// compiled to 44.  A point's 8 planes are 64 bytes of LDS, read as four
// 16-byte broadcasts for the thread's HPT = 2 targets.  Each of the
// block's 4 waves holds the tile's 128 targets and takes every fourth
// pencil; the waves' sums are added in wave order.  With 256 targets a block
// and every wave its own 64 (the form before) N = 100k had 1.5 waves per
// SIMD.  N = 500k, degree 5, 7.3e9 pairs: 13.6 -> 6.7 ms (7.8 with tiles of
// 256 targets on pairs of waves); N = 100k 4.5 -> 2.1 ms; Yukawa with
// subtraction, N = 100k, degree 4: 5.6 -> 3.5 ms.
// ---------------------------------------------------------------------
constexpr int HPT = 2;                // targets per thread
constexpr int HPTS = 256;             // points per LDS chunk (whole pencils)
static_assert(HERM_PC_TILE == 64 * HPT && HTPB == 256, "a wave's targets, four waves");

// the forms of planes c in the displacement: linear, bilinear, trilinear
// (yz = dy dz)
__device__ __forceinline__ void herm_forms(const double *c, double dx, double dy, double dz, double yz, double &lin,
                                           double &bil, double &tri)
{
    lin = fma(c[3], dz, fma(c[2], dy, c[1] * dx));
    bil = fma(dx, fma(c[6], dz, c[4] * dy), c[5] * yz);
    tri = (c[7] * yz) * dx;
}

// One point's expansion: dyz2 = dy^2 + dz^2 (r2 = dx^2 + dyz2).  Coulomb and
// regularized Coulomb planes 4..6 come multiplied by 3, plane 7 by 15.
template <int KER, bool SS>
__device__ __forceinline__ void herm_pc_pair(double dx, double dy, double dz, double dyz2, double yz, const double *q,
                                             const double *w, double tq, const KParams &kp, const double *tab,
                                             double &acc)
{
    double r2 = fma(dx, dx, dyz2);
    if constexpr (KER == HKS) {
        // derivative expansion of sin(k r)/r; coincident points are skipped
        // (sin-over-r_pc.c:68-155)
        const double k = kp.p0, k2 = k * k, k3 = k * k2;
        const double r = sqrt(r2);
        if (!(r > DBL_MIN)) return;
        const double rinv = 1.0 / r;
        const double r2inv = rinv * rinv, r3inv = rinv * r2inv, r4inv = r2inv * r2inv;
        const double r5inv = r3inv * r2inv, r6inv = r3inv * r3inv, r7inv = r4inv * r3inv;
        double sn, cs;
        sincos(k * r, &sn, &cs);
        acc += sn * rinv * q[0] + (sn * r3inv - k * cs * r2inv) * (q[1] * dx + q[2] * dy + q[3] * dz) +
               (sn * (3 * r5inv - k2 * r3inv) - 3 * k * cs * r4inv) *
                   (q[4] * dx * dy + q[5] * dy * dz + q[6] * dx * dz) +
               (sn * (15 * r7inv - 6 * k2 * r5inv) + cs * (k3 * r4inv - 15 * k * r6inv)) * q[7] * dx * dy * dz;
    } else if constexpr (KER == HKY) {
        // e^{-x} (c0 + (1+x) L/r^2 + (3+3x+x^2) B/r^4 + (15+15x+6x^2+x^3) T/r^6)/r, x = k r
        const double ir = rsq64(r2), i2 = ir * ir, r = r2 * ir, x = kp.p0 * r;
        double c[8], lin, bil, tri;
#pragma unroll
        for (int m = 0; m < 8; m++) c[m] = SS ? fma(-w[m], tq, q[m]) : q[m];
        herm_forms(c, dx, dy, dz, yz, lin, bil, tri);
        const double p3 = fma(x, fma(x, x + 6.0, 15.0), 15.0), p2 = fma(x, x + 3.0, 3.0);
        double s = fma(i2 * p3, tri, p2 * bil);
        s = fma(i2, s, fma(x, lin, lin));
        s = fma(i2, s, c[0]);
        acc = fma(exp_neg(r, kp.ek, tab) * ir, s, acc);
    } else {
        // Coulomb and regularized Coulomb: (q0 + L/r^2 + 3 B/r^4 + 15 T/r^6)/r
        // (r with eps^2 for the regularized kernel); subtraction adds the
        // expansion of e^{-r^2/k^2}/r weighted by -tq
        if constexpr (KER == HKR) r2 += kp.eps2;
        const double ir = rsq64(r2), i2 = ir * ir;
        const double lin = fma(q[3], dz, fma(q[2], dy, q[1] * dx));
        const double u = fma(i2, q[7] * yz, fma(q[6], dz, q[4] * dy));
        double s = fma(i2, fma(dx, u, q[5] * yz), lin);
        s = fma(i2, s, q[0]);
        if constexpr (SS) {
            double lw, bw, tw;
            herm_forms(w, dx, dy, dz, yz, lw, bw, tw);
            const double x = r2 * kp.inv_a2;
            const double p3 = fma(x, fma(x, fma(x, 8.0, 12.0), 18.0), 15.0);
            const double p2 = fma(x, fma(x, 4.0, 4.0), 3.0), p1 = fma(x, 2.0, 1.0);
            double sw = fma(i2 * p3, tw, p2 * bw);
            sw = fma(i2, sw, p1 * lw);
            sw = fma(i2, sw, w[0]);
            s = fma(-tq * exp_neg(r2, kp.eg, tab), sw, s);
        }
        acc = fma(ir, s, acc);
    }
}

template <int KER, bool SS>
__global__ __launch_bounds__(HTPB) void k_herm_pc(HermPCArgs a)
{
    constexpr bool EXPS = KER == HKY || (SS && KER != HKS);
    const Tile tile = a.tiles[blockIdx.x];
    if (tile.z == 0) return;
    const int tid = threadIdx.x;
    const int nl = a.nl, P = nl * nl * nl, n2 = nl * nl;
    __shared__ alignas(16) double Lq[HPTS][8];
    __shared__ alignas(16) double Lw[SS ? HPTS : 1][8];
    __shared__ double Lt[3 * (MAX_DEGREE + 1)];  // the cluster's Chebyshev points
    __shared__ double Ltab[EXPS ? EXP_TAB : 1];
    __shared__ double Lr[4][HERM_PC_TILE];  // the waves' sums
    if constexpr (EXPS) exp_table(Ltab, tid);
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    int ix[HPT];
    double tx[HPT], ty[HPT], tz[HPT], tq[HPT], acc[HPT];
#pragma unroll
    for (int u = 0; u < HPT; u++) {
        const int li = lane + 64 * u;
        ix[u] = tile.y + (li < tile.z ? li : 0);
        tx[u] = a.tx[ix[u]]; ty[u] = a.ty[ix[u]]; tz[u] = a.tz[ix[u]];
        tq[u] = SS ? a.tq[ix[u]] : 0.0;
        acc[u] = 0.0;
    }
    const int pens = HPTS / nl;  // pencils per chunk
    for (int c = a.clu_off[tile.x]; c < a.clu_off[tile.x + 1]; c++) {
        const size_t node = (size_t)a.clu_id[c];
        const double *cq = a.cq + node * 8 * P;
        const double *cw = SS ? a.cw + node * 8 * P : nullptr;
        for (int pb = 0; pb < n2; pb += pens) {
            const int np = min(pens, n2 - pb), n = np * nl;
            __syncthreads();  // the previous chunk has been read
            if (tid < 3 * nl) Lt[tid] = a.tab[node * 3 * nl + tid];
            if (tid < n) {
                const int j = tid;
#pragma unroll
                for (int m = 0; m < 8; m++) {
                    // 3 and 15 of the Coulomb expansion
                    constexpr bool C = KER == HKC || KER == HKR;
                    const double f = C && m == 7 ? 15.0 : (C && m >= 4 ? 3.0 : 1.0);
                    Lq[j][m] = f * cq[m * P + pb * nl + j];
                    if constexpr (SS) Lw[j][m] = cw[m * P + pb * nl + j];
                }
            }
            __syncthreads();
            int k2 = (pb + wv) % nl, k3 = (pb + wv) / nl;
            for (int pen = wv; pen < np; pen += 4) {
                double dy[HPT], dz[HPT], dyz2[HPT], yz[HPT];
#pragma unroll
                for (int u = 0; u < HPT; u++) {
                    dy[u] = ty[u] - Lt[nl + k2];
                    dz[u] = tz[u] - Lt[2 * nl + k3];
                    dyz2[u] = fma(dz[u], dz[u], dy[u] * dy[u]);
                    yz[u] = dy[u] * dz[u];
                }
                for (int k1 = 0; k1 < nl; k1++) {
                    const int j = pen * nl + k1;
                    const double x = Lt[k1];
                    double q[8], w[8];
#pragma unroll
                    for (int m = 0; m < 8; m++) {
                        q[m] = Lq[j][m];
                        w[m] = SS ? Lw[SS ? j : 0][m] : 0.0;
                    }
#pragma unroll
                    for (int u = 0; u < HPT; u++)
                        herm_pc_pair<KER, SS>(tx[u] - x, dy[u], dz[u], dyz2[u], yz[u], q, w, tq[u], a.kp, Ltab, acc[u]);
                }
                k2 += 4;
                while (k2 >= nl) { k2 -= nl; k3++; }
            }
        }
    }
#pragma unroll
    for (int u = 0; u < HPT; u++) Lr[wv][lane + 64 * u] = acc[u];
    __syncthreads();
    if (tid < tile.z) a.pot[tile.y + tid] += ((Lr[0][tid] + Lr[1][tid]) + Lr[2][tid]) + Lr[3][tid];
}

// ---------------------------------------------------------------------
// Cluster-particle far field: tile {key, first grid point, count, node} of
// up to HTPB grid points of a target node against the source ranges of its
// key; the 8 plane sums go to the key's output row (coulomb_cp.c:66-184,
// yukawa_cp.c:68-194, regularized-coulomb_cp.c:68-188,
// sin-over-r_cp.c:68-198).  A tile of at most HTPB/2 points leaves room for
// G = HTPB / count shares of the sources: thread (share, point) takes every
// G-th source and the shares' sums are added in share order, so the grids of
// degrees 1 to 4 (8 to 125 points) fill the block.  Coulomb: 28 FP64
// instructions per pair (the expressions as the reference writes them
// compiled to about 34): the second derivatives' common factor is applied once,
// and 3 and 15 after the sums.  N = 500k, degree 5: 10.7 -> 9.2 ms; N = 100k,
// degree 3 (64 points): 3.1 -> 0.7 ms.
// ---------------------------------------------------------------------
template <int KER>
__global__ __launch_bounds__(HTPB) void k_herm_cp(HermCPArgs a)
{
    const Tile tile = a.tiles[blockIdx.x];
    if (tile.z == 0) return;
    const int tid = threadIdx.x;
    const int nl = a.nl, P = nl * nl * nl;
    __shared__ double4 Ls[HTPB];
    __shared__ double Lr[HTPB];
    __shared__ double Ltab[KER == HKY ? EXP_TAB : 1];
    if constexpr (KER == HKY) exp_table(Ltab, tid);
    const int G = HTPB / tile.z;  // shares of the sources (1 above HTPB/2 points)
    const int share = tid / tile.z, lp = tid - share * tile.z;
    const bool on = share < G;
    const int jl = tile.y + lp;
    const int k1 = jl % nl, k2 = (jl / nl) % nl, k3 = jl / (nl * nl);
    const double *tab = a.tab + (size_t)tile.w * 3 * nl;
    const double cx = tab[k1], cy = tab[nl + k2], cz = tab[2 * nl + k3];
    double t[8];
#pragma unroll
    for (int m = 0; m < 8; m++) t[m] = 0.0;
    for (int s = a.seg_off[tile.x]; s < a.seg_off[tile.x + 1]; s++) {
        const Seg sg = a.segs[s];
        const int cnt = (int)((unsigned)sg.y & SEG_COUNT_MASK);
        for (int off = 0; off < cnt; off += HTPB) {
            const int n = min(HTPB, cnt - off);
            __syncthreads();
            if (tid < n) {
                const int g = sg.x + off + tid;
                Ls[tid] = make_double4(a.sx[g], a.sy[g], a.sz[g], a.sq[g]);
            }
            __syncthreads();
            if (!on) continue;
            for (int jj = share; jj < n; jj += G) {
                const double4 S = Ls[jj];
                const double dx = S.x - cx, dy = S.y - cy, dz = S.z - cz;
                double r2 = fma(dz, dz, fma(dy, dy, dx * dx));
                if constexpr (KER == HKS) {
                    const double k = a.kp.p0, k2 = k * k, k3 = k * k2;
                    const double r = sqrt(r2);
                    const double rinv = 1.0 / r;
                    const double r2inv = rinv * rinv, r3inv = rinv * r2inv, r4inv = r2inv * r2inv;
                    const double r5inv = r3inv * r2inv, r6inv = r3inv * r3inv, r7inv = r4inv * r3inv;
                    double sn, cs;
                    sincos(k * r, &sn, &cs);
                    sn *= S.w; cs *= S.w;
                    const double d1 = sn * r3inv - k * cs * r2inv;
                    const double d2 = sn * (3 * r5inv - k2 * r3inv) - 3 * k * cs * r4inv;
                    const double d3 = sn * (15 * r7inv - 6 * k2 * r5inv) + cs * (k3 * r4inv - 15 * k * r6inv);
                    t[0] += sn * rinv;
                    t[1] += d1 * dx; t[2] += d1 * dy; t[3] += d1 * dz;
                    t[4] += d2 * dx * dy; t[5] += d2 * dy * dz; t[6] += d2 * dx * dz;
                    t[7] += d3 * dx * dy * dz;
                } else {
                    if constexpr (KER == HKR) r2 += a.kp.eps2;
                    const double ir = rsq64(r2), i2 = ir * ir;
                    // g q; the factors of the first, second and third
                    // derivatives d1, d2, d3 (Coulomb: over 1, 3, 15)
                    double g, d1, d2, d3;
                    if constexpr (KER == HKY) {
                        const double r = r2 * ir, x = a.kp.p0 * r;
                        g = S.w * ir * exp_neg(r, a.kp.ek, Ltab);
                        const double g3 = g * i2, g5 = g3 * i2;
                        d1 = fma(g3, x, g3);
                        d2 = g5 * fma(x, x + 3.0, 3.0);
                        d3 = g5 * i2 * fma(x, fma(x, x + 6.0, 15.0), 15.0);
                    } else {
                        g = S.w * ir;
                        d1 = g * i2;
                        d2 = d1 * i2;
                        d3 = 0.0;
                    }
                    t[0] += g;
                    t[1] = fma(d1, dx, t[1]); t[2] = fma(d1, dy, t[2]); t[3] = fma(d1, dz, t[3]);
                    const double d2y = d2 * dy, d2xy = d2y * dx;
                    t[4] += d2xy;
                    t[5] = fma(d2y, dz, t[5]);
                    t[6] = fma(d2 * dx, dz, t[6]);
                    t[7] = fma(KER == HKY ? d3 * dx * dy : d2xy * i2, dz, t[7]);
                }
            }
        }
    }
    if constexpr (KER == HKC || KER == HKR) {
        t[4] *= 3.0; t[5] *= 3.0; t[6] *= 3.0;
        t[7] *= 15.0;
    }
    double *o = a.rows + a.out_row[tile.x];
#pragma unroll
    for (int m = 0; m < 8; m++) {
        if (G > 1) {  // block-uniform
            __syncthreads();
            Lr[tid] = t[m];
            __syncthreads();
            if (share == 0)
                for (int q = 1; q < G; q++) t[m] += Lr[q * tile.z + lp];
        }
        if (share == 0) o[(size_t)m * P + jl] = t[m];
    }
}

// One node's 8-plane interpolant at the thread's target p (the node's
// Chebyshev nodes and Hermite weights in Lnode/Lw; planes q).
template <int NL>
__device__ double herm_down_node(const double p[3], const double (*Lnode)[NL], const double (*Lw)[NL],
                                 double (*Lq)[NL * NL], const double *q, int tid)
{
    constexpr int n = NL - 1, P = NL * NL * NL, S = NL * NL;
    // factors per dimension; exact hits (downpass.c:962-975)
    double A[3][NL], B[3][NL];
    double den = 1.0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        int e = -1;
        double sum = 0.0;
#pragma unroll
        for (int k = 0; k < NL; k++) {
            const double dx = p[d] - Lnode[d][k];
            if (fabs(dx) < DBL_MIN) e = k;
            const double dj = herm_dj(k, n);
            A[d][k] = dj / (dx * dx) + Lw[d][k] / dx;
            B[d][k] = dj / dx;
            sum += A[d][k];
        }
        if (e == -1) {
            den /= sum;
        } else {
#pragma unroll
            for (int k = 0; k < NL; k++) { A[d][k] = k == e ? 1.0 : 0.0; B[d][k] = 0.0; }
        }
    }
    double temp = 0.0;
#pragma unroll 1
    for (int k3 = 0; k3 < NL; k3++) {
        __syncthreads();
        for (int g = tid; g < 8 * S; g += HTPB) Lq[g / S][g % S] = q[(size_t)(g / S) * P + k3 * S + g % S];
        __syncthreads();
        double az = 0.0, bz = 0.0;
#pragma unroll
        for (int k = 0; k < NL; k++)
            if (k == k3) { az = A[2][k]; bz = B[2][k]; }
#pragma unroll
        for (int k2 = 0; k2 < NL; k2++) {
            const double yz00 = A[1][k2] * az, yz10 = B[1][k2] * az, yz01 = A[1][k2] * bz, yz11 = B[1][k2] * bz;
#pragma unroll
            for (int k1 = 0; k1 < NL; k1++) {
                const int j = k2 * NL + k1;
                const double va = yz00 * Lq[0][j] + yz10 * Lq[2][j] + yz01 * Lq[3][j] + yz11 * Lq[5][j];
                const double vb = yz00 * Lq[1][j] + yz10 * Lq[4][j] + yz01 * Lq[6][j] + yz11 * Lq[7][j];
                temp = fma(A[0][k1], va, fma(B[0][k1], vb, temp));
            }
        }
    }
    return den * temp;
}

// ---------------------------------------------------------------------
// Downpass: tile {leaf, first target, count} of up to HTPB targets (one per
// thread).  Every node containing a target adds its 8-plane interpolant to
// it (interaction_compute_downpass.c:117-120, 860-1109); here a target
// walks from its leaf to the root, summing the interpolants of the nodes
// that received planes, and adds the sum once (no two blocks touch one
// target).  A node's planes stream through LDS one z-slab (8 x NL^2 values)
// at a time.
// ---------------------------------------------------------------------
template <int NL>
__global__ __launch_bounds__(HTPB) void k_herm_down(HermDownArgs a)
{
    constexpr int P = NL * NL * NL, S = NL * NL;
    const Tile tile = a.tiles[blockIdx.x];
    if (tile.z == 0) return;
    const int tid = threadIdx.x;
    __shared__ double Lnode[3][NL], Lw[3][NL];
    __shared__ double Lq[8][S];
    const int i = tile.y + (tid < tile.z ? tid : 0);
    const double p[3] = {a.tx[i], a.ty[i], a.tz[i]};
    double total = 0.0;
    for (int node = tile.x; node >= 0; node = a.parent[node]) {
        if (a.rows_off[node + 1] == a.rows_off[node]) continue;  // no planes (uniform in the block)
        __syncthreads();
        if (tid < 3 * NL) {
            Lnode[tid / NL][tid % NL] = a.tab[(size_t)node * 3 * NL + tid];
            Lw[tid / NL][tid % NL] = a.wtab[(size_t)node * 3 * NL + tid];
        }
        __syncthreads();
        total += herm_down_node<NL>(p, Lnode, Lw, Lq, a.Q + (size_t)node * 8 * P, tid);
    }
    if (tid < tile.z) a.pot[i] += total;
}


template <bool SS>
hipError_t herm_anterp_dispatch(const HermAnterpArgs &a, hipStream_t st)
{
    const int nl = a.degree + 1, P = nl * nl * nl;
    dim3 g(a.nparts, (P + HTPB - 1) / HTPB), b(HTPB);
    switch (a.degree) {
#define CASE(D) case D: k_herm_anterp<D + 1, SS><<<g, b, 0, st>>>(a); break;
        CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11) CASE(12)
#undef CASE
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_herm_anterp(const HermAnterpArgs &a, hipStream_t st)
{
    if (a.nparts <= 0) return hipSuccess;
    return a.subtraction ? herm_anterp_dispatch<true>(a, st) : herm_anterp_dispatch<false>(a, st);
}

hipError_t launch_herm_pc(const HermPCArgs &a, hipStream_t st)
{
    if (a.ntiles <= 0) return hipSuccess;
    if (a.nl < 2 || a.nl > MAX_DEGREE + 1) return hipErrorInvalidValue;
    dim3 g(a.ntiles), b(HTPB);
    const bool ss = a.singularity == 2;
#define L(K, S) k_herm_pc<K, S><<<g, b, 0, st>>>(a)
    switch (a.kernel) {
        case HKC: if (ss) L(HKC, true); else L(HKC, false); break;
        case HKY: if (ss) L(HKY, true); else L(HKY, false); break;
        case HKR: if (ss) L(HKR, true); else L(HKR, false); break;
        case HKS: if (ss) return hipErrorInvalidValue; L(HKS, false); break;
        default: return hipErrorInvalidValue;
    }
#undef L
    return hipGetLastError();
}

hipError_t launch_herm_cp(const HermCPArgs &a, hipStream_t st)
{
    if (a.ntiles <= 0) return hipSuccess;
    dim3 g(a.ntiles), b(HTPB);
    switch (a.kernel) {
        case HKC: k_herm_cp<HKC><<<g, b, 0, st>>>(a); break;
        case HKY: k_herm_cp<HKY><<<g, b, 0, st>>>(a); break;
        case HKR: k_herm_cp<HKR><<<g, b, 0, st>>>(a); break;
        case HKS: k_herm_cp<HKS><<<g, b, 0, st>>>(a); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_herm_down(const HermDownArgs &a, hipStream_t st)
{
    if (a.ntiles <= 0) return hipSuccess;
    dim3 g(a.ntiles), b(HTPB);
    switch (a.degree) {
#define CASE(D) case D: k_herm_down<D + 1><<<g, b, 0, st>>>(a); break;
        CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11) CASE(12)
#undef CASE
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace btk
