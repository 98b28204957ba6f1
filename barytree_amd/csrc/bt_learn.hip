// bt_learn.hip -- gfx950 kernels of the learned degree selection:
//   k_label            : minimal degree of a far-field pair (FP64, one block per pair)
//   k_mlp_infer        : MLP forward and degrees from the logits (FP32)
//   k_mlp_grad         : forward, loss, backward and partial weight gradients
//   k_mlp_sum          : the partial gradients' sum
//   k_mlp_adam         : the sum and the Adam update
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>

#include "bt_exp.h"
#include "bt_learn.h"
#include "bt_rsq.h"

namespace btl {

namespace {

// ---------------------------------------------------------------------
// Pair labels.  One block of 4 waves per pair; degrees are tried in order.
// A degree's heavy part is a sum over points (sources, or source grid points)
// for each of a set of grid points; its work items are (grid point, share of
// the points): G = label_split shares per grid point, so that the small grids
// of the low degrees fill the block too, the shares added in order
// afterwards.  FP64; 1/r by rsq64, exponentials from the table of bt_exp.h.
// Instantiated per kind, kernel and singularity, so that a block holds only
// the arrays its kind uses: 34 kB of LDS for a cluster-particle pair (4
// blocks per CU), where one kernel for every kind held 128 kB (1 block, one
// wave per SIMD) and took IEEE square roots and divisions and three integer
// divisions per term.  16k cluster-particle pairs of a 300k Plummer sphere
// (regularized Coulomb, tol 1e-7, 190k terms a pair): 18.5 -> 2.5 ms, of which
// the terms' 17 FP64 instructions each take 1.7.
// ---------------------------------------------------------------------
constexpr int LTPB = 256;
constexpr int NLMAX = LABEL_DMAX + 1;
constexpr int PMAX = NLMAX * NLMAX * NLMAX;
constexpr int LPT = LTPB / LABEL_NT;  // lanes per sampled target (8)
constexpr int L_PC = 1, L_CP = 2;     // pair kinds (3: CC)

// Shares of the points per grid point of degree nl - 1: what leaves the
// fewest of the block's threads and steps idle for 128 points (at least
// 0.87 busy), within PMAX partial sums.
__device__ __forceinline__ int label_split(int nl)
{
    switch (nl) {
        case 3: return 9;
        case 4: return 8;
        case 5: return 8;
        case 6: return 7;
        case 7: return 5;
        case 8: return 2;
        default: return 1;
    }
}

// (k1, k2, k3) of grid point j = k1 + nl (k2 + nl k3); exact for j < 4096,
// nl <= 13: the quotient's error j (ceil(2^16/nl) - 2^16/nl) / 2^16 is below
// j / 2^16 < 1/nl
__device__ __forceinline__ void grid_index(int j, int nl, int &k1, int &k2, int &k3)
{
    const unsigned m = (65536u + nl - 1) / nl;
    const int r = (int)(((unsigned)j * m) >> 16);
    k1 = j - r * nl;
    k3 = (int)(((unsigned)r * m) >> 16);
    k2 = r - k3 * nl;
}

// The pair's kernel from r^2 (1/r, e^{-kappa r}/r, 1/sqrt(r^2 + eps^2)), and
// with subtraction the second term's, which multiplies the source weight
// and, at the target, minus the target's charge (coulomb_ss_pc.c:47,
// yukawa_ss_pc.c:46, regularized-coulomb_ss_pc.c, coulomb_ss_cp.c:54-55):
// Coulomb e^{-r^2/k^2}/r, Yukawa the same kernel, regularized Coulomb
// e^{-r^2/a^2}/sqrt(r^2 + eps^2)
struct LabelKernel {
    double eps2;
    btk::ExpRate ek, eg;
    const double *tab;
};

template <int KER, bool SS>
__device__ __forceinline__ void green(const LabelKernel &K, double r2, double a, double b, double &v, double &vw)
{
    const double ir = btk::rsq64(KER == 3 ? r2 + K.eps2 : r2);
    if constexpr (KER == 2) {
        const double g = btk::exp_neg(r2 * ir, K.ek, K.tab) * ir;
        v = fma(a, g, v);
        if constexpr (SS) vw = fma(b, g, vw);
    } else {
        v = fma(a, ir, v);
        if constexpr (SS) vw = fma(b, btk::exp_neg(r2, K.eg, K.tab) * ir, vw);
    }
}

// Lagrange basis at Chebyshev points (barycentric form, second kind):
// l_k(x) = (w_k/(x-x_k)) / sum_j w_j/(x-x_j), w_k = (-1)^k d_k with
// d_0 = d_n = 1/2; an exact hit |x - x_k| < DBL_MIN gives the Kronecker row.
__device__ void lagrange_row(double x, const double *nodes, int nl, double *out)
{
    const int n = nl - 1;
    double sum = 0.0;
    int hit = -1;
    for (int k = 0; k < nl; k++) {
        const double c = x - nodes[k];
        if (fabs(c) < DBL_MIN) hit = k;
        const double d = (k == 0 || k == n) ? 0.5 : 1.0;
        const double v = ((k & 1) ? -d : d) / c;
        out[k] = v;
        sum += v;
    }
    for (int k = 0; k < nl; k++) out[k] = hit >= 0 ? (k == hit ? 1.0 : 0.0) : out[k] / sum;
}

// sum over the LPT lanes of a group (lanes tid & ~(LPT-1) .. +LPT-1), fixed order
__device__ __forceinline__ double group_sum(double v)
{
#pragma unroll
    for (int o = LPT / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, LPT);
    return v;
}

template <int KIND, int KER, bool SS>
__global__ __launch_bounds__(LTPB) void k_label(LabelArgs A, LabelKernel K)
{
    constexpr int NT = LABEL_NT, NS = LABEL_NS;
    constexpr bool SRC = KIND != L_CP, TGT = KIND != L_PC;  // interpolated sides
    constexpr bool EXPS = SS || KER == 2;
    const int pi = blockIdx.x, tid = threadIdx.x;
    if (A.kind[pi] != KIND) return;  // another instantiation's (block-uniform)

    __shared__ double4 Ls[NS];  // sources: x, y, z, first term's charge
    __shared__ double Lsw[SS ? NS : 1];
    __shared__ double Ltx[NT], Lty[NT], Ltz[NT], Ltq[NT], Lex[NT], Lred[2 * NT];
    __shared__ double Lnt[3 * NLMAX], Lns[3 * NLMAX];
    __shared__ double Bs[SRC ? NS * 3 * NLMAX : 1];
    __shared__ double Bt[TGT ? NT * 3 * NLMAX : 1];
    // grid values of the two terms (the second only with subtraction)
    __shared__ double G1[SRC ? PMAX : 1], G1w[SRC && SS ? PMAX : 1];
    // (CC: in the place of the source basis, which has been read by then)
    __shared__ double G2s[TGT && !SRC ? (SS ? 2 : 1) * PMAX : 1];
    static_assert(NS * 3 * NLMAX >= 2 * PMAX, "target grids fit the source basis");
    double *const G2 = SRC ? Bs : G2s, *const G2w = G2 + PMAX;
    __shared__ double Ltab[EXPS ? btk::EXP_TAB : 1];
    if constexpr (EXPS) btk::exp_table(Ltab, tid);
    K.tab = Ltab;

    const int tb0 = A.tbeg[pi], tc = A.tcnt[pi], sb0 = A.sbeg[pi], sc = A.scnt[pi];
    const int nt = min(tc, NT), ns = min(sc, NS);
    const double *tbox = A.tbox + 6 * (size_t)pi, *sbox = A.sbox + 6 * (size_t)pi;
    if (tid < nt) {
        const int i = tb0 + (int)(((long long)tid * tc) / nt);
        Ltx[tid] = A.tx[i]; Lty[tid] = A.ty[i]; Ltz[tid] = A.tz[i];
        Ltq[tid] = SS ? A.tq[i] : 0.0;
    }
    if (tid < ns) {
        const int s = sb0 + (int)(((long long)tid * sc) / ns);
        // subtraction: the first term's charge is q w, the second's w
        double q = A.sq[s];
        if constexpr (SS) {
            const double w = A.sw[s];
            Lsw[tid] = w;
            q *= w;
        }
        Ls[tid] = make_double4(A.sx[s], A.sy[s], A.sz[s], q);
    }
    __syncthreads();

    const int g = tid / LPT, l = tid % LPT;  // target of this lane group, lane in group
    const double tx = g < nt ? Ltx[g] : 0.0, ty = g < nt ? Lty[g] : 0.0, tz = g < nt ? Ltz[g] : 0.0;
    // exact sums at the sampled targets
    {
        double v = 0.0, vw = 0.0;
        if (g < nt)
            for (int s = l; s < ns; s += LPT) {
                const double4 p = Ls[s];
                const double dx = tx - p.x, dy = ty - p.y, dz = tz - p.z;
                green<KER, SS>(K, fma(dz, dz, fma(dy, dy, dx * dx)), p.w, SS ? Lsw[s] : 0.0, v, vw);
            }
        v = group_sum(v);
        if constexpr (SS) vw = group_sum(vw);
        if (l == 0 && g < nt) Lex[g] = SS ? v - Ltq[g] * vw : v;
    }

    int label = LABEL_DMAX + 1;
    for (int p = LABEL_DMIN; p <= LABEL_DMAX; p++) {
        const int nl = p + 1, n2 = nl * nl, P = n2 * nl, G = label_split(nl);
        __syncthreads();  // the previous degree's arrays have been read
        if (tid < 3 * nl) {
            const int d = tid / nl, k = tid % nl;
            const double u = (cos(k * M_PI / p) + 1.0) * 0.5;
            Lnt[d * nl + k] = tbox[2 * d] + u * (tbox[2 * d + 1] - tbox[2 * d]);
            Lns[d * nl + k] = sbox[2 * d] + u * (sbox[2 * d + 1] - sbox[2 * d]);
        }
        __syncthreads();
        if constexpr (SRC)
            for (int i = tid; i < ns * 3; i += LTPB) {
                const int s = i / 3, d = i % 3;
                const double c = d == 0 ? Ls[s].x : (d == 1 ? Ls[s].y : Ls[s].z);
                lagrange_row(c, Lns + d * nl, nl, Bs + i * NLMAX);
            }
        if constexpr (TGT)
            for (int i = tid; i < nt * 3; i += LTPB) {
                const int t = i / 3, d = i % 3;
                const double c = d == 0 ? Ltx[t] : (d == 1 ? Lty[t] : Ltz[t]);
                lagrange_row(c, Lnt + d * nl, nl, Bt + i * NLMAX);
            }
        // the shares' sums (X[g P + j]) added in order into X[j]
        auto combine = [&](double *X, double *Xw) {
            __syncthreads();
            if (G > 1) {
                for (int j = tid; j < P; j += LTPB) {
                    double v = X[j], vw = SS ? Xw[j] : 0.0;
                    for (int q = 1; q < G; q++) {
                        v += X[q * P + j];
                        if constexpr (SS) vw += Xw[q * P + j];
                    }
                    X[j] = v;
                    if constexpr (SS) Xw[j] = vw;
                }
                __syncthreads();
            }
        };
        if constexpr (SRC) {
            __syncthreads();
            // modified charges of the source grid: Q_k = sum_s q_s l_k(y_s)
            for (int it = tid; it < P * G; it += LTPB) {
                const int q = it / P, j = it - q * P;
                int k1, k2, k3;
                grid_index(j, nl, k1, k2, k3);
                double v = 0.0, vw = 0.0;
#pragma unroll 2
                for (int s = q; s < ns; s += G) {
                    const double *r = Bs + 3 * s * NLMAX;
                    const double b = r[k1] * r[NLMAX + k2] * r[2 * NLMAX + k3];
                    v = fma(Ls[s].w, b, v);
                    if constexpr (SS) vw = fma(Lsw[s], b, vw);
                }
                G1[it] = v;
                if constexpr (SS) G1w[it] = vw;
            }
            combine(G1, G1w);
        }
        if constexpr (TGT) {
            // target grid values, from the sources (CP) or the source grid (CC)
            if constexpr (!SRC) __syncthreads();
            for (int it = tid; it < P * G; it += LTPB) {
                const int q = it / P, j = it - q * P;
                int k1, k2, k3;
                grid_index(j, nl, k1, k2, k3);
                const double gx = Lnt[k1], gy = Lnt[nl + k2], gz = Lnt[2 * nl + k3];
                double v = 0.0, vw = 0.0;
                if constexpr (KIND == L_CP) {
#pragma unroll 4
                    for (int s = q; s < ns; s += G) {
                        const double4 c = Ls[s];
                        const double dx = gx - c.x, dy = gy - c.y, dz = gz - c.z;
                        green<KER, SS>(K, fma(dz, dz, fma(dy, dy, dx * dx)), c.w, SS ? Lsw[s] : 0.0, v, vw);
                    }
                } else {
                    // the source grid's pencils (m2, m3) of the share
                    int m2 = q % nl, m3 = q / nl;
                    for (int m = q; m < n2; m += G) {
                        const double dy = gy - Lns[nl + m2], dz = gz - Lns[2 * nl + m3];
                        const double dyz = fma(dz, dz, dy * dy);
                        for (int m1 = 0; m1 < nl; m1++) {
                            const double dx = gx - Lns[m1];
                            green<KER, SS>(K, fma(dx, dx, dyz), G1[m * nl + m1], SS ? G1w[m * nl + m1] : 0.0, v, vw);
                        }
                        m2 += G;
                        while (m2 >= nl) { m2 -= nl; m3++; }
                    }
                }
                G2[it] = v;
                if constexpr (SS) G2w[it] = vw;
            }
            combine(G2, G2w);
        }
        // approximation at the sampled targets: the group's lanes take the
        // pencils (m2, m3) of the grid in turn
        double v = 0.0, vw = 0.0;
        if (g < nt) {
            int m2 = l % nl, m3 = l / nl;
            const double *b = Bt + (TGT ? g * 3 * NLMAX : 0);
            for (int m = l; m < n2; m += LPT) {
                if constexpr (KIND == L_PC) {
                    const double dy = ty - Lns[nl + m2], dz = tz - Lns[2 * nl + m3];
                    const double dyz = fma(dz, dz, dy * dy);
                    for (int m1 = 0; m1 < nl; m1++) {
                        const double dx = tx - Lns[m1];
                        green<KER, SS>(K, fma(dx, dx, dyz), G1[m * nl + m1], SS ? G1w[m * nl + m1] : 0.0, v, vw);
                    }
                } else {
                    const double f = b[NLMAX + m2] * b[2 * NLMAX + m3];
                    double x = 0.0, xw = 0.0;
                    for (int m1 = 0; m1 < nl; m1++) {
                        x = fma(b[m1], G2[m * nl + m1], x);
                        if constexpr (SS) xw = fma(b[m1], G2w[m * nl + m1], xw);
                    }
                    v = fma(f, x, v);
                    if constexpr (SS) vw = fma(f, xw, vw);
                }
                m2 += LPT;
                while (m2 >= nl) { m2 -= nl; m3++; }
            }
        }
        v = group_sum(v);
        if constexpr (SS) vw = group_sum(vw);
        if (l == 0) {
            const double e = g < nt ? (SS ? v - Ltq[g] * vw : v) - Lex[g] : 0.0;
            Lred[g] = e * e;
            Lred[NT + g] = g < nt ? Lex[g] * Lex[g] : 0.0;
        }
        __syncthreads();
        // every thread forms the same two sums
        double num = 0.0, den = 0.0;
        for (int i = 0; i < NT; i++) { num += Lred[i]; den += Lred[NT + i]; }
        // a sampled point on another's place makes the sums NaN (rsq64(0)):
        // the error is NaN then, which no tolerance accepts
        const double err = num == 0.0 && den == 0.0 ? 0.0 : sqrt(num / den);
        if (tid == 0) A.errors[(size_t)pi * LABEL_ND + (p - LABEL_DMIN)] = err;
        if (err <= A.tol) { label = p; break; }  // block-uniform
    }
    if (tid == 0) {
        A.labels[pi] = label;
        for (int p = label + 1; p <= LABEL_DMAX; p++)
            A.errors[(size_t)pi * LABEL_ND + (p - LABEL_DMIN)] = NAN;
    }
}

template <int KER, bool SS>
hipError_t label_dispatch(const LabelArgs &a, const LabelKernel &k, hipStream_t st)
{
    // every kind over the whole list, each block keeping the pairs of its own
    k_label<1, KER, SS><<<a.npairs, LTPB, 0, st>>>(a, k);
    k_label<2, KER, SS><<<a.npairs, LTPB, 0, st>>>(a, k);
    k_label<3, KER, SS><<<a.npairs, LTPB, 0, st>>>(a, k);
    return hipGetLastError();
}

// ---------------------------------------------------------------------
// MLP, FP32 on the matrix cores (v_mfma_f32_16x16x4f32: FP32 operands,
// products and sums).  A block of 4 waves takes tiles of MS = 32 samples;
// activations and gradients live in LDS feature-major, H[f][s] with rows of
// MSP = 33 floats, and the weights in registers: wave w owns output rows
// 16w .. 16w+15 of every 64-wide product and keeps their weights (and the
// transposed ones of the backward pass) for all its tiles.  Lane l holds
//   A[l%16][k], B[k][l%16] for k = KQ (l/16) + step,  KQ = K/4,
//   D[4 (l/16) + v][l%16], v = 0..3
// (any assignment of k to lanes and steps serves, as long as A and B agree:
// this one makes a lane's weights consecutive in memory, and puts the four
// lane groups' rows of H in different LDS banks).
//
// The whole pass over a batch -- normalisation, three hidden layers, output,
// loss, backward and the weight gradients of the block's samples, kept in
// the accumulators over its tiles -- is one launch; the blocks' partial
// gradients are added in block order by the launch that applies Adam.  A
// training step is bound by latency (4096 samples need 2.3e8 flops): 14
// launches, four of them weight gradients on at most 20 blocks (174 us each),
// and a copy of the losses after each step took 1.03 ms a step at batch 4096;
// two launches (16 and 4 us) and no copy take 21 us (24 steps: 24.7 -> 2.3 ms with
// the call's own host work).
// ---------------------------------------------------------------------
constexpr int MTPB = 256, MWAVES = 4;
constexpr int MS = MLP_TILE;   // samples per tile
constexpr int MSP = MS + 1;    // 16 MSP = 16 mod 64 banks
constexpr int MCT = MS / 16;   // column tiles of 16 samples
static_assert(MLP_H == 16 * MWAVES && MS == 32 && MLP_OUT <= 16 && MLP_IN == 8, "MLP layout");

typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float sigmoidf_(float z) { return 1.0f / (1.0f + expf(-z)); }

// this lane's weights of rows r0 .. r0+15 of W (rows x K, row major); rows
// outside give zeros
template <int K>
__device__ __forceinline__ void load_rows(const float *W, int r0, int rows, int lane, float (&a)[K / 4])
{
    const int r = r0 + (lane & 15);
    const float *p = W + (size_t)(r < rows ? r : 0) * K + (K / 4) * (lane >> 4);
#pragma unroll
    for (int s = 0; s < K / 4; s++) a[s] = r < rows ? p[s] : 0.0f;
}

// rows c0 .. c0+15 of W^T, W being rows x cols row major, K >= rows
template <int K>
__device__ __forceinline__ void load_cols(const float *W, int c0, int rows, int cols, int lane, float (&a)[K / 4])
{
    const int c = c0 + (lane & 15);
#pragma unroll
    for (int s = 0; s < K / 4; s++) {
        const int r = (K / 4) * (lane >> 4) + s;
        a[s] = r < rows ? W[(size_t)r * cols + c] : 0.0f;
    }
}

// D += A B for columns 16 ct .. of H (K rows)
template <int K>
__device__ __forceinline__ v4f product(const float (&a)[K / 4], const float *H, int ct, int lane, v4f d)
{
    const float *h = H + (K / 4) * (lane >> 4) * MSP + 16 * ct + (lane & 15);
#pragma unroll
    for (int s = 0; s < K / 4; s++) d = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], h[s * MSP], d, 0, 0, 0);
    return d;
}

// D += X[16 xr ..][samples] Y[16 yr ..][samples]^T over the tile's samples
__device__ __forceinline__ v4f outer(const float *X, int xr, const float *Y, int yr, int lane, v4f d)
{
    const int o = (lane & 15) * MSP + (MS / 4) * (lane >> 4);
    const float *x = X + 16 * xr * MSP + o, *y = Y + 16 * yr * MSP + o;
#pragma unroll
    for (int s = 0; s < MS / 4; s++) d = __builtin_amdgcn_mfma_f32_16x16x4f32(x[s], y[s], d, 0, 0, 0);
    return d;
}

// the hidden layers' and the output's weights and biases of a wave
struct MlpForward {
    float w1[MLP_IN / 4], w2[MLP_H / 4], w3[MLP_H / 4], w4[MLP_H / 4];
    v4f b1, b2, b3, b4;
    __device__ __forceinline__ void load(const float *prm, int wv, int lane)
    {
        load_rows<MLP_IN>(prm + OFF_W1, 16 * wv, MLP_H, lane, w1);
        load_rows<MLP_H>(prm + OFF_W2, 16 * wv, MLP_H, lane, w2);
        load_rows<MLP_H>(prm + OFF_W3, 16 * wv, MLP_H, lane, w3);
        load_rows<MLP_H>(prm + OFF_W4, 0, MLP_OUT, lane, w4);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int r = 4 * (lane >> 4) + v;
            b1[v] = prm[OFF_B1 + 16 * wv + r];
            b2[v] = prm[OFF_B2 + 16 * wv + r];
            b3[v] = prm[OFF_B3 + 16 * wv + r];
            b4[v] = r < MLP_OUT ? prm[OFF_B4 + r] : 0.0f;
        }
    }
};

// rows 16 wv .. of Hout = relu(A Hin + bias)
template <int K>
__device__ __forceinline__ void hidden(const float (&a)[K / 4], v4f bias, const float *Hin, float *Hout, int wv,
                                       int lane)
{
#pragma unroll
    for (int ct = 0; ct < MCT; ct++) {
        const v4f d = product<K>(a, Hin, ct, lane, bias);
#pragma unroll
        for (int v = 0; v < 4; v++)
            Hout[(16 * wv + 4 * (lane >> 4) + v) * MSP + 16 * ct + (lane & 15)] = fmaxf(d[v], 0.0f);
    }
}

// rows 16 wv .. of G = [H > 0] (A D)
template <int K>
__device__ __forceinline__ void backward(const float (&a)[K / 4], const float *D, const float *H, float *G, int wv,
                                         int lane)
{
#pragma unroll
    for (int ct = 0; ct < MCT; ct++) {
        const v4f d = product<K>(a, D, ct, lane, v4f{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int o = (16 * wv + 4 * (lane >> 4) + v) * MSP + 16 * ct + (lane & 15);
            G[o] = H[o] > 0.0f ? d[v] : 0.0f;
        }
    }
}

// normalised inputs of the tile's samples, H0[f][s] (zero past the batch):
// thread 8 s + f
__device__ __forceinline__ void inputs(const float *x, const int *idx, const float *mean, const float *scale, int s0,
                                       int nb, float *H0)
{
    const int f = threadIdx.x & (MLP_IN - 1), s = threadIdx.x / MLP_IN;
    const int b = s0 + s;
    float v = 0.0f;
    if (b < nb) v = (x[(size_t)(idx ? idx[b] : b) * MLP_IN + f] - mean[f]) * scale[f];
    H0[f * MSP + s] = v;
}

__global__ __launch_bounds__(MTPB) void k_mlp_grad(const float *prm, const float *mean, const float *scale,
                                                   const float *x, const int *labels, const int *idx, int nb,
                                                   float *part, double *loss)
{
    __shared__ float H0[16 * MSP], H1[MLP_H * MSP], H2[MLP_H * MSP], H3[MLP_H * MSP];
    __shared__ float D1[MLP_H * MSP], D2[MLP_H * MSP], D3[MLP_H * MSP], DZ[16 * MSP];
    __shared__ double Ll[2 * 64];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const float inv_b = 1.0f / (float)nb;
    MlpForward w;
    w.load(prm, wv, lane);
    float t2[MLP_H / 4], t3[MLP_H / 4], t4[16 / 4];
    load_cols<MLP_H>(prm + OFF_W2, 16 * wv, MLP_H, MLP_H, lane, t2);
    load_cols<MLP_H>(prm + OFF_W3, 16 * wv, MLP_H, MLP_H, lane, t3);
    load_cols<16>(prm + OFF_W4, 16 * wv, MLP_OUT, MLP_H, lane, t4);
    // rows 8.. of H0 are only read by the gradient of W1, whose columns 8..
    // are not stored; row 8 holds ones: column 8 is the bias gradient
    for (int e = tid; e < 8 * MSP; e += MTPB) H0[8 * MSP + e] = e < MSP ? 1.0f : 0.0f;
    const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
    v4f g1 = zero, g2[4], g3[4], g4 = zero;
#pragma unroll
    for (int c = 0; c < 4; c++) { g2[c] = zero; g3[c] = zero; }
    // bias gradients: thread i of D2's rows, then D3's, then DZ's
    float gb = 0.0f;
    double lsum = 0.0;
    for (int s0 = blockIdx.x * MS; s0 < nb; s0 += gridDim.x * MS) {
        __syncthreads();  // the previous tile has been read
        inputs(x, idx, mean, scale, s0, nb, H0);
        __syncthreads();
        hidden<MLP_IN>(w.w1, w.b1, H0, H1, wv, lane);
        __syncthreads();
        hidden<MLP_H>(w.w2, w.b2, H1, H2, wv, lane);
        __syncthreads();
        hidden<MLP_H>(w.w3, w.b3, H2, H3, wv, lane);
        __syncthreads();
        if (wv < MCT) {
            // logits of column tile wv, loss and output gradient
            const int s = 16 * wv + (lane & 15), b = s0 + s;
            const bool on = b < nb;
            const int lab = on ? labels[idx ? idx[b] : b] : 0;
            const v4f z4 = product<MLP_H>(w.w4, H3, wv, lane, w.b4);
            float l = 0.0f;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int k = 4 * (lane >> 4) + v;
                const float z = z4[v], y = lab > LABEL_DMIN + k ? 1.0f : 0.0f;
                const bool use = on && k < MLP_OUT;
                if (use) l += fmaxf(z, 0.0f) + log1pf(expf(-fabsf(z))) - y * z;
                DZ[k * MSP + s] = use ? (sigmoidf_(z) - y) * inv_b : 0.0f;
            }
            lsum += (double)l;
        }
        __syncthreads();
        backward<16>(t4, DZ, H3, D3, wv, lane);
        __syncthreads();
        backward<MLP_H>(t3, D3, H2, D2, wv, lane);
        __syncthreads();
        backward<MLP_H>(t2, D2, H1, D1, wv, lane);
        __syncthreads();
        g1 = outer(D1, wv, H0, 0, lane, g1);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            g2[c] = outer(D2, wv, H1, c, lane, g2[c]);
            g3[c] = outer(D3, wv, H2, c, lane, g3[c]);
        }
        g4 = outer(DZ, 0, H3, wv, lane, g4);
        const float *d = tid < MLP_H ? D2 + tid * MSP
                       : tid < 2 * MLP_H ? D3 + (tid - MLP_H) * MSP
                       : tid < 2 * MLP_H + MLP_OUT ? DZ + (tid - 2 * MLP_H) * MSP : nullptr;
        if (d)
            for (int s = 0; s < MS; s++) gb += d[s];
    }
    // this block's row of partial gradients
    float *o = part + (size_t)blockIdx.x * MLP_PARAMS;
    const int col = lane & 15;
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int r = 4 * (lane >> 4) + v, i = 16 * wv + r;
        if (col < MLP_IN) o[OFF_W1 + i * MLP_IN + col] = g1[v];
        else if (col == MLP_IN) o[OFF_B1 + i] = g1[v];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            o[OFF_W2 + i * MLP_H + 16 * c + col] = g2[c][v];
            o[OFF_W3 + i * MLP_H + 16 * c + col] = g3[c][v];
        }
        if (r < MLP_OUT) o[OFF_W4 + r * MLP_H + 16 * wv + col] = g4[v];
    }
    if (tid < MLP_H) o[OFF_B2 + tid] = gb;
    else if (tid < 2 * MLP_H) o[OFF_B3 + tid - MLP_H] = gb;
    else if (tid < 2 * MLP_H + MLP_OUT) o[OFF_B4 + tid - 2 * MLP_H] = gb;
    if (wv < MCT) Ll[tid] = lsum;
    __syncthreads();
    if (tid == 0) {
        double s = 0.0;
        for (int k = 0; k < 64 * MCT; k++) s += Ll[k];
        loss[blockIdx.x] = s;
    }
}

// Logits (sample major, optional) and degrees (optional) of n samples.
__global__ __launch_bounds__(MTPB) void k_mlp_infer(const float *prm, const float *mean, const float *scale,
                                                    const float *x, int n, float delta, float *logits, int *degree)
{
    __shared__ float H0[MLP_IN * MSP], HA[MLP_H * MSP], HB[MLP_H * MSP], Z[MS * MLP_OUT];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    MlpForward w;
    w.load(prm, wv, lane);
    for (int s0 = blockIdx.x * MS; s0 < n; s0 += gridDim.x * MS) {
        __syncthreads();
        inputs(x, nullptr, mean, scale, s0, n, H0);
        __syncthreads();
        hidden<MLP_IN>(w.w1, w.b1, H0, HA, wv, lane);
        __syncthreads();
        hidden<MLP_H>(w.w2, w.b2, HA, HB, wv, lane);
        __syncthreads();
        hidden<MLP_H>(w.w3, w.b3, HB, HA, wv, lane);
        __syncthreads();
        if (wv < MCT) {
            const v4f z4 = product<MLP_H>(w.w4, HA, wv, lane, w.b4);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int k = 4 * (lane >> 4) + v;
                if (k < MLP_OUT) Z[(16 * wv + (lane & 15)) * MLP_OUT + k] = z4[v];
            }
        }
        __syncthreads();
        const int m = min(MS, n - s0);
        if (logits)
            for (int e = tid; e < m * MLP_OUT; e += MTPB) logits[(size_t)s0 * MLP_OUT + e] = Z[e];
        if (degree && tid < m) {
            int deg = LABEL_DMIN;
#pragma unroll
            for (int k = 0; k < MLP_OUT; k++)
                if (sigmoidf_(Z[tid * MLP_OUT + k]) >= delta) deg = LABEL_DMIN + 1 + k;
            degree[s0 + tid] = deg;
        }
    }
}

// The blocks' rows in block order, four runs of them side by side and then
// in order: the gradient (grad) or one Adam step with it.
constexpr int RPB = 64;  // parameters per block
__device__ __forceinline__ bool reduced(const float *part, int nparts, int &i, float &g)
{
    __shared__ float L[4][RPB];
    const int c = threadIdx.x % RPB, q = threadIdx.x / RPB;
    i = blockIdx.x * RPB + c;
    float s = 0.0f;
    if (i < MLP_PARAMS) {
        const int e = nparts * (q + 1) / 4;
#pragma unroll 8
        for (int k = nparts * q / 4; k < e; k++) s += part[(size_t)k * MLP_PARAMS + i];
    }
    L[q][c] = s;
    __syncthreads();
    g = ((L[0][c] + L[1][c]) + L[2][c]) + L[3][c];
    return q == 0 && i < MLP_PARAMS;
}

__global__ __launch_bounds__(4 * RPB) void k_mlp_sum(const float *part, int nparts, float *grad)
{
    int i;
    float g;
    if (reduced(part, nparts, i, g)) grad[i] = g;
}

__global__ __launch_bounds__(4 * RPB) void k_mlp_adam(const float *part, int nparts, float *p, float *m, float *v,
                                                      float lr, float b1, float b2, float eps, float c1, float c2)
{
    int i;
    float gi;
    if (!reduced(part, nparts, i, gi)) return;
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

}  // namespace

hipError_t launch_label(const LabelArgs &a, hipStream_t st)
{
    if (a.npairs <= 0) return hipSuccess;
    LabelKernel k{};
    k.eps2 = a.p0 * a.p0;
    k.ek = btk::exp_rate(a.p0);
    k.eg = btk::exp_rate(a.p1);
    switch (a.kernel) {
        case 1: return a.ss ? label_dispatch<1, true>(a, k, st) : label_dispatch<1, false>(a, k, st);
        case 2: return a.ss ? label_dispatch<2, true>(a, k, st) : label_dispatch<2, false>(a, k, st);
        case 3: return a.ss ? label_dispatch<3, true>(a, k, st) : label_dispatch<3, false>(a, k, st);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_mlp_infer(const float *params, const float *mean, const float *scale, int n,
                            const float *x, float delta, float *logits, int *degree, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    const int tiles = (n + MS - 1) / MS;
    k_mlp_infer<<<tiles < 2048 ? tiles : 2048, MTPB, 0, st>>>(params, mean, scale, x, n, delta, logits, degree);
    return hipGetLastError();
}

hipError_t launch_mlp_grad(const float *params, const float *mean, const float *scale, const float *x,
                           const int *labels, const int *idx, int b, float *part, double *loss, hipStream_t st)
{
    if (b <= 0) return hipSuccess;
    k_mlp_grad<<<mlp_parts(b), MTPB, 0, st>>>(params, mean, scale, x, labels, idx, b, part, loss);
    return hipGetLastError();
}

hipError_t launch_mlp_sum(const float *part, int nparts, float *grad, hipStream_t st)
{
    k_mlp_sum<<<(MLP_PARAMS + RPB - 1) / RPB, 4 * RPB, 0, st>>>(part, nparts, grad);
    return hipGetLastError();
}

hipError_t launch_mlp_adam(const float *part, int nparts, float *params, float *m, float *v, float lr,
                           float beta1, float beta2, float eps, int t, hipStream_t st)
{
    const float c1 = 1.0f / (1.0f - powf(beta1, (float)t));
    const float c2 = 1.0f / (1.0f - powf(beta2, (float)t));
    k_mlp_adam<<<(MLP_PARAMS + RPB - 1) / RPB, 4 * RPB, 0, st>>>(part, nparts, params, m, v, lr, beta1, beta2, eps,
                                                                 c1, c2);
    return hipGetLastError();
}

}  // namespace btl
