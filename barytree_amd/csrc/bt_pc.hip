// bt_pc.hip -- particle targets against source clusters in FP64, the clusters
// as tensor grids (K_*_PC_Lagrange and the subtraction forms).
//
// The NL^3 points of a source cluster are (x_a, y_b, z_c), so for one target
// r^2 = (t_x - x_a)^2 + [(t_y - y_b)^2 + (t_z - z_c)^2]: the NL squares of the
// x displacements are formed once per cluster and kept in registers, the
// bracket once per pencil (b, c), and a pair costs one addition before the
// kernel (r^2 summed as dx^2 + (dz^2 + dy^2), a few ulp of r^2 from the
// reference's order) where the particle launch took three subtractions, a
// product and two fma, and one 8-byte charge from LDS instead of 32 bytes of
// coordinates and charge.  Tiles of 64 PCT targets; each of a block's 4 waves
// holds all of them (PCT per thread) and takes every fourth pencil, so a few
// thousand targets fill the chip; the waves' sums are added in wave order.
// Every target's sum has one order whatever the tiles around it.
//
// Coulomb, the whole execution beside the symmetric near field: N = 100k,
// degree 8 (1.9e9 pairs) 4.1 -> 3.0 ms; N = 200k, degree 12, 20 -> 11.8 ms;
// Yukawa N = 300k, degree 6, 21.5 -> 15.8 ms.
//
// The subtraction's Gaussian of Coulomb and regularized Coulomb is a product
// over the dimensions (SEP): NL factors e^{-dx^2/a^2} per target and cluster
// and one factor of y and z per target and pencil, so a pair pays two
// products for an 11-instruction exponential: Coulomb N = 200k, degree 7,
// 11.9 -> 9.9 ms; N = 100k, degree 12 (bound by its near field) 7.7 -> 7.6.
#include <hip/hip_runtime.h>

#include "bt_kernels.h"
#include "bt_pair.h"

namespace btk {
namespace {

constexpr int PTPB = 256, PCT = 2;  // threads per block, targets per thread
static_assert(PC_TILE == 64 * PCT, "a wave's targets");

template <int KER, bool SS, int NL>
__global__ __launch_bounds__(PTPB) void k_pc64(PcArgs A)
{
    constexpr int P = NL * NL * NL, N2 = NL * NL;
    constexpr bool SEP = separable_gauss(KER, SS);
    constexpr int PENS = P <= 1024 ? N2 : 1024 / NL;  // pencils staged at a time
    __shared__ double Lq[PENS * NL], Lw[SS ? PENS * NL : 1];
    __shared__ double Lt[3 * NL];
    __shared__ double Lr[4][PC_TILE];
    __shared__ alignas(16) double Ltab[pair_table_len(KER, SS)];
    const Tile tile = A.tiles[blockIdx.x];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    pair_table<KER, SS>(Ltab, tid, PTPB);  // read after the first staging barrier
    double tx[PCT], ty[PCT], tz[PCT], tq[PCT], acc[PCT];
#pragma unroll
    for (int u = 0; u < PCT; u++) {
        const int li = lane + 64 * u;
        const int i = tile.y + (li < tile.z ? li : 0);
        tx[u] = A.tx[i]; ty[u] = A.ty[i]; tz[u] = A.tz[i];
        tq[u] = SS ? A.tq[i] : 0.0;
        acc[u] = 0.0;
    }
    const int c1 = A.clu_off[tile.x + 1];
    for (int c = A.clu_off[tile.x]; c < c1; c++) {
        const size_t node = (size_t)A.clu_id[c];
        double dx2[PCT][NL], ex[PCT][SEP ? NL : 1];
        for (int pb = 0; pb < N2; pb += PENS) {
            const int np = min(PENS, N2 - pb);
            __syncthreads();  // the previous pencils have been read
            if (tid < 3 * NL) Lt[tid] = A.tab[node * 3 * NL + tid];
            for (int j = tid; j < np * NL; j += PTPB) {
                Lq[j] = A.cq[node * P + pb * NL + j];
                if constexpr (SS) Lw[j] = A.cw[node * P + pb * NL + j];
            }
            __syncthreads();
            if (pb == 0)
#pragma unroll
                for (int u = 0; u < PCT; u++)
#pragma unroll
                    for (int k = 0; k < NL; k++) {
                        const double dx = tx[u] - Lt[k];
                        dx2[u][k] = dx * dx;
                        if constexpr (SEP) ex[u][k] = exp_neg(dx2[u][k], A.kp.eg, Ltab);
                    }
            for (int pen = wv; pen < np; pen += 4) {
                const int k3 = (pb + pen) / NL, k2 = pb + pen - k3 * NL;
                const double y = Lt[NL + k2], z = Lt[2 * NL + k3];
                double dyz2[PCT], eyz[PCT];
#pragma unroll
                for (int u = 0; u < PCT; u++) {
                    const double dy = ty[u] - y, dz = tz[u] - z;
                    dyz2[u] = fma(dz, dz, dy * dy);
                    eyz[u] = SEP ? -tq[u] * exp_neg(dyz2[u], A.kp.eg, Ltab) : 0.0;
                    if constexpr (SEP && KER == KR) dyz2[u] += A.kp.eps2;
                }
#pragma unroll
                for (int k = 0; k < NL; k++) {
                    const double q = Lq[pen * NL + k], w = SS ? Lw[pen * NL + k] : 0.0;
#pragma unroll
                    for (int u = 0; u < PCT; u++)
                        if constexpr (SEP)
                            acc[u] = fma(fma(eyz[u] * ex[u][k], w, q), rsq64(dx2[u][k] + dyz2[u]), acc[u]);
                        else
                            pair_r2<KER, SS, false, true>(dx2[u][k] + dyz2[u], q, w, tq[u], A.kp, acc[u], Ltab);
                }
            }
        }
    }
#pragma unroll
    for (int u = 0; u < PCT; u++) Lr[wv][lane + 64 * u] = acc[u];
    __syncthreads();
    if (tid < tile.z) A.pot[tile.y + tid] += ((Lr[0][tid] + Lr[1][tid]) + Lr[2][tid]) + Lr[3][tid];
}

template <int KER, bool SS>
hipError_t pc_dispatch(const PcArgs &a, hipStream_t st)
{
    switch (a.nl) {
#define CASE(NL) case NL: k_pc64<KER, SS, NL><<<a.ntiles, PTPB, 0, st>>>(a); break;
        CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8) CASE(9) CASE(10) CASE(11) CASE(12) CASE(13)
#undef CASE
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_pc64(const PcArgs &a, hipStream_t st)
{
    if (a.ntiles <= 0) return hipSuccess;
    const bool ss = a.singularity == 2;
    switch (a.kernel) {
        case KC: return ss ? pc_dispatch<KC, true>(a, st) : pc_dispatch<KC, false>(a, st);
        case KY: return ss ? pc_dispatch<KY, true>(a, st) : pc_dispatch<KY, false>(a, st);
        case KR: return ss ? pc_dispatch<KR, true>(a, st) : pc_dispatch<KR, false>(a, st);
        case KRY: return ss ? pc_dispatch<KRY, true>(a, st) : pc_dispatch<KRY, false>(a, st);
        case KSR: return ss ? hipErrorInvalidValue : pc_dispatch<KSR, false>(a, st);
        case KUS: return ss ? hipErrorInvalidValue : pc_dispatch<KUS, false>(a, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace btk
