// First derivatives of the two-electron energy, one quartet per lane: the
// classes whose two-particle density block and three 2D tables (one more unit
// of angular momentum on i, j and k) fit the registers; the others run on the
// runtime-l kernel of jk_generic.hip.
//
// The survivors are found as in jk_lane_kernel (jk_class_kernels.h), one
// wavefront per work item.  Per primitive quartet and root a lane builds the
// tables of x, y and z and adds, for every element n of the block,
//   Gamma_n g_x(i_x + 1) g_y g_z   and   -i_x Gamma_n g_x(i_x - 1) g_y g_z
// (likewise y, z and the centres j, k): the first sums are scaled by 2 a_i
// once per primitive quartet, so no derivative table is formed and an element
// costs 6 multiplications and 9 to 18 FMAs.  The sums of i and j are kept in
// registers over the whole work item; those of k and l (by translational
// invariance) are added to the atoms per quartet.
// Bound by latency at one or two waves per SIMD (tables in 140-512 registers).
// Gradient of 4 water molecules (def2-SVP): every class on the runtime-l kernel
// 61.4 ms, the small ones here 6.6 ms.
#include "jk_launch.h"

// doubles of Gamma and the three tables
#define IP1_LANE_MAX 200

template <int LI, int LJ, int LK, int LL>
struct Ip1Lane {
    static constexpr int NF = ncart(LI) * ncart(LJ) * ncart(LK) * ncart(LL);
    static constexpr int GS = (LI + 2) * (LJ + 2) * (LK + 2) * (LL + 1);
    static constexpr bool ON = NF + 3 * GS <= IP1_LANE_MAX;
};

// One quartet: adds its derivatives with respect to i, j and k to gi, gj, gk.
template <int LI, int LJ, int LK, int LL>
__device__ __forceinline__ void ip1_quartet(double *gi, double *gj, double *gk,
                                            const double *gamma, const JKBuildArgs &a,
                                            const ShellPair &sp, const double *pij, int nij,
                                            const double *pkl, int nkl, const double *rk,
                                            const double *rkl, const double *expk, double omega2,
                                            const lds_double *rows)
{
    constexpr int NFI = ncart(LI), NFJ = ncart(LJ), NFK = ncart(LK), NFL = ncart(LL);
    constexpr int N = (LI + LJ + LK + LL + 1) / 2 + 1;
    constexpr int GS = Ip1Lane<LI, LJ, LK, LL>::GS;
    constexpr int SK = LL + 1, SJ = (LK + 2) * SK, SI = (LJ + 2) * SJ;
    constexpr CartPow<LI> ci{};
    constexpr CartPow<LJ> cj{};
    constexpr CartPow<LK> ck{};
    constexpr CartPow<LL> cl{};
    const double *ei = a.env + sp.pexpi, *ej = a.env + sp.pexpj;
    for (int kp = 0; kp < nkl; ++kp) {
        const double *q = pkl + kp * PREC;
        const double akl = q[0], rakl = q[1];
        const double QC[3] = {q[2] - rk[0], q[3] - rk[1], q[4] - rk[2]};
        const double ak2 = 2. * expk[kp / a.lprim];
        for (int ip = 0; ip < nij; ++ip) {
            const double *p = pij + ip * PREC;
            const double aij = p[0], raij = p[1];
            double PA[3], PQ[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                PA[d] = p[2 + d] - sp.ri[d];
                PQ[d] = p[2 + d] - q[2 + d];
            }
            const double rr = PQ[0]*PQ[0] + PQ[1]*PQ[1] + PQ[2]*PQ[2];
            const double r_aa = rcp64(aij + akl);
            const double theta = aij * akl * r_aa;
            const double fac = p[5] * q[5] * rsqrt64(aij + akl);
            double aw = 1., sa = 1.;
            if (omega2 > 0.) {          // long-range attenuation (see eri_lane)
                aw = omega2 / (omega2 + theta);
                sa = sqrt(aw);
            }
            double rt[N], wt[N];
            rys_roots<N>(a.rys, rows, theta * rr * aw, rt, wt);
            double ui[3] = {0., 0., 0.}, uj[3] = {0., 0., 0.}, uk[3] = {0., 0., 0.};
#pragma unroll
            for (int r = 0; r < N; ++r) {
                const double rt_aa = rt[r] * aw * r_aa;
                const double rt_aij = rt_aa * akl, rt_akl = rt_aa * aij;
                const double b10 = .5 * raij * (1. - rt_aij);
                const double b01 = .5 * rakl * (1. - rt_akl);
                const double b00 = .5 * rt_aa;
                double gx[GS], gy[GS], gz[GS];
                build_g<LI + 1, LJ + 1, LK + 1, LL>(gx, 1., PA[0] - rt_aij * PQ[0],
                                                    QC[0] + rt_akl * PQ[0], b10, b01, b00,
                                                    sp.rij[0], rkl[0]);
                build_g<LI + 1, LJ + 1, LK + 1, LL>(gy, 1., PA[1] - rt_aij * PQ[1],
                                                    QC[1] + rt_akl * PQ[1], b10, b01, b00,
                                                    sp.rij[1], rkl[1]);
                build_g<LI + 1, LJ + 1, LK + 1, LL>(gz, wt[r] * sa * fac, PA[2] - rt_aij * PQ[2],
                                                    QC[2] + rt_akl * PQ[2], b10, b01, b00,
                                                    sp.rij[2], rkl[2]);
#pragma unroll
                for (int i = 0; i < NFI; ++i)
#pragma unroll
                for (int j = 0; j < NFJ; ++j)
#pragma unroll
                for (int k = 0; k < NFK; ++k)
#pragma unroll
                for (int l = 0; l < NFL; ++l) {
                    const int ox = ci.x[i]*SI + cj.x[j]*SJ + ck.x[k]*SK + cl.x[l];
                    const int oy = ci.y[i]*SI + cj.y[j]*SJ + ck.y[k]*SK + cl.y[l];
                    const int oz = ci.z[i]*SI + cj.z[j]*SJ + ck.z[k]*SK + cl.z[l];
                    const double g = gamma[((i*NFJ + j)*NFK + k)*NFL + l];
                    const double wx = g * gx[ox], wy = g * gy[oy];
                    const double yz = wy * gz[oz], xz = wx * gz[oz], xy = wx * gy[oy];
                    ui[0] = fma(yz, gx[ox + SI], ui[0]);
                    ui[1] = fma(xz, gy[oy + SI], ui[1]);
                    ui[2] = fma(xy, gz[oz + SI], ui[2]);
                    uj[0] = fma(yz, gx[ox + SJ], uj[0]);
                    uj[1] = fma(xz, gy[oy + SJ], uj[1]);
                    uj[2] = fma(xy, gz[oz + SJ], uj[2]);
                    uk[0] = fma(yz, gx[ox + SK], uk[0]);
                    uk[1] = fma(xz, gy[oy + SK], uk[1]);
                    uk[2] = fma(xy, gz[oz + SK], uk[2]);
                    if (ci.x[i]) gi[0] = fma(-ci.x[i] * yz, gx[ox - SI], gi[0]);
                    if (ci.y[i]) gi[1] = fma(-ci.y[i] * xz, gy[oy - SI], gi[1]);
                    if (ci.z[i]) gi[2] = fma(-ci.z[i] * xy, gz[oz - SI], gi[2]);
                    if (cj.x[j]) gj[0] = fma(-cj.x[j] * yz, gx[ox - SJ], gj[0]);
                    if (cj.y[j]) gj[1] = fma(-cj.y[j] * xz, gy[oy - SJ], gj[1]);
                    if (cj.z[j]) gj[2] = fma(-cj.z[j] * xy, gz[oz - SJ], gj[2]);
                    if (ck.x[k]) gk[0] = fma(-ck.x[k] * yz, gx[ox - SK], gk[0]);
                    if (ck.y[k]) gk[1] = fma(-ck.y[k] * xz, gy[oy - SK], gk[1]);
                    if (ck.z[k]) gk[2] = fma(-ck.z[k] * xy, gz[oz - SK], gk[2]);
                }
            }
            const double ai2 = 2. * ei[ip / a.jprim], aj2 = 2. * ej[ip % a.jprim];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                gi[d] = fma(ai2, ui[d], gi[d]);
                gj[d] = fma(aj2, uj[d], gj[d]);
                gk[d] = fma(ak2, uk[d], gk[d]);
            }
        }
    }
}

template <int LI, int LJ, int LK, int LL>
__global__ __launch_bounds__(WAVE)
void jk_ip1_lane_kernel(JKBuildArgs a, TaskBatch batch, GenExtra ex)
{
    constexpr int NFI = ncart(LI), NFJ = ncart(LJ), NFK = ncart(LK), NFL = ncart(LL);
    constexpr int N = (LI + LJ + LK + LL + 1) / 2 + 1;
    __shared__ uint32_t queue[2 * WAVE];
    __shared__ __align__(16) double moment_buf[MomentRows<N>::SIZE];
    const lds_double *rows = (const lds_double *)moment_buf;
    int kl_chunk, unused;
    const int item = select_task(a, batch, kl_chunk, unused);
    const int lane = threadIdx.x;
    const int nbas = a.nbas, nao = a.nao;
    if (a.n_repl > 1) ex.ejk += (int64_t)(blockIdx.x % a.n_repl) * a.repl_stride;
    const WorkItem wi = work_item(item, a.npairs_kl, kl_chunk);
    const uint32_t bas_ij = a.pairs_ij[wi.pij];
    const float kl_cutoff = a.cutoff - a.q_ij[wi.pij];
    if (a.q_kl[wi.kl0] + Q_COND_MARGIN < kl_cutoff) return;
    const bool do_j = ex.jf != 0., do_k = ex.kf != 0.;
    ShellPair sp;
    load_shell_pair(sp, bas_ij, nbas, a.bas, a.env, a.ao_loc);
    const int i0 = sp.i0, j0 = sp.j0;
    const int nij = a.iprim * a.jprim, nkl = a.kprim * a.lprim;
    const double *pij = a.pdata_ij + (size_t)wi.pij * nij * PREC;
    const double omega2 = a.omega * a.omega;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    load_moment_rows<N>(moment_buf, a.rys, lane, WAVE);
    __syncthreads();
    double gij[6];
#pragma unroll
    for (int t = 0; t < 6; ++t) gij[t] = 0.;
    int qn = 0;
    unsigned long long nsurv = 0, hsum = 0;
    bool stop = false;
    for (int base = wi.kl0; base < wi.kl1 || qn > 0; base += WAVE) {
        if (base < wi.kl1 && !stop) {
            const int pkl = base + lane;
            bool keep = false, fail_margin = false;
            if (pkl < wi.kl1) {
                const float q_kl = a.q_kl[pkl];
                const uint32_t bkl = a.pairs_kl[pkl];
                fail_margin = q_kl + Q_COND_MARGIN < kl_cutoff;
                keep = survives_ejk(q_kl, kl_cutoff, bas_ij, bkl, sp.ish, sp.jsh, nbas,
                                    a.dm_cond, do_j, do_k);
                if (a.quartet_hash && keep) hsum += quartet_mix(bas_ij, bkl);
            }
            const uint64_t m = __ballot(keep);
            if (keep) queue[qn + __popcll(m & lt_mask)] = pkl;
            qn += __popcll(m);
            nsurv += __popcll(m);
            stop = __ballot(fail_margin) != 0;
            wave_sync();
        }
        const bool flush = base + WAVE >= wi.kl1 || stop;
        if (qn >= WAVE || (flush && qn > 0)) {
            const int nb = min(qn, WAVE);
            const bool active = lane < nb;
            const int pkl = queue[active ? lane : 0];
            const uint32_t bas_kl = a.pairs_kl[pkl];
            const int ksh = bas_kl / nbas, lsh = bas_kl - (bas_kl / nbas) * nbas;
            double fac_sym = a.scale;
            if (sp.ish == sp.jsh) fac_sym *= .5;
            if (ksh == lsh) fac_sym *= .5;
            if (bas_ij == bas_kl) fac_sym *= .5;
            if (!active) fac_sym = 0.;
            const int k0 = a.ao_loc[ksh], l0 = a.ao_loc[lsh];
            // two-particle density of the block (rys_contract_jk_ip1.cu:523-577)
            double gamma[NFI * NFJ * NFK * NFL];
            {
                double dij[NFI * NFJ], dkl[NFK * NFL];
#pragma unroll
                for (int n = 0; n < NFI * NFJ; ++n) dij[n] = 0.;
#pragma unroll
                for (int n = 0; n < NFK * NFL; ++n) dkl[n] = 0.;
#pragma unroll
                for (int n = 0; n < NFI * NFJ * NFK * NFL; ++n) gamma[n] = 0.;
                for (int id = 0; id < a.n_dm; ++id) {
                    const double *D = a.dm + (size_t)id * nao * nao;
                    double dik[NFI * NFK], dil[NFI * NFL], djk[NFJ * NFK], djl[NFJ * NFL];
#pragma unroll
                    for (int k = 0; k < NFK; ++k) {
                        const double *row = D + (size_t)(k0 + k) * nao;
#pragma unroll
                        for (int i = 0; i < NFI; ++i) dik[i*NFK + k] = row[i0 + i];
#pragma unroll
                        for (int j = 0; j < NFJ; ++j)
                            djk[j*NFK + k] = D[(size_t)(j0 + j) * nao + k0 + k];
                    }
#pragma unroll
                    for (int l = 0; l < NFL; ++l) {
                        const double *row = D + (size_t)(l0 + l) * nao;
#pragma unroll
                        for (int i = 0; i < NFI; ++i) dil[i*NFL + l] = row[i0 + i];
#pragma unroll
                        for (int j = 0; j < NFJ; ++j)
                            djl[j*NFL + l] = D[(size_t)(j0 + j) * nao + l0 + l];
#pragma unroll
                        for (int k = 0; k < NFK; ++k) dkl[k*NFL + l] += row[k0 + k];
                    }
#pragma unroll
                    for (int i = 0; i < NFI; ++i)
#pragma unroll
                    for (int j = 0; j < NFJ; ++j)
                        dij[i*NFJ + j] += D[(size_t)(j0 + j) * nao + i0 + i];
#pragma unroll
                    for (int i = 0; i < NFI; ++i)
#pragma unroll
                    for (int j = 0; j < NFJ; ++j)
#pragma unroll
                    for (int k = 0; k < NFK; ++k)
#pragma unroll
                    for (int l = 0; l < NFL; ++l)
                        gamma[((i*NFJ + j)*NFK + k)*NFL + l] +=
                            djk[j*NFK + k] * dil[i*NFL + l] + djl[j*NFL + l] * dik[i*NFK + k];
                }
                const double kf = ex.kf * fac_sym, jf = ex.jf * fac_sym;
#pragma unroll
                for (int i = 0; i < NFI; ++i)
#pragma unroll
                for (int j = 0; j < NFJ; ++j)
#pragma unroll
                for (int k = 0; k < NFK; ++k)
#pragma unroll
                for (int l = 0; l < NFL; ++l) {
                    const int n = ((i*NFJ + j)*NFK + k)*NFL + l;
                    gamma[n] = kf * gamma[n] + jf * dij[i*NFJ + j] * dkl[k*NFL + l];
                }
            }
            const double *rk = a.env + a.bas[ksh * 8 + 7], *rl = a.env + a.bas[lsh * 8 + 7];
            const double rk3[3] = {rk[0], rk[1], rk[2]};
            const double rkl[3] = {rl[0] - rk[0], rl[1] - rk[1], rl[2] - rk[2]};
            double gi[3] = {0., 0., 0.}, gj[3] = {0., 0., 0.}, gk[3] = {0., 0., 0.};
            ip1_quartet<LI, LJ, LK, LL>(gi, gj, gk, gamma, a, sp, pij, nij,
                                        a.pdata_kl + (size_t)pkl * nkl * PREC, nkl, rk3, rkl,
                                        a.env + a.bas[ksh * 8 + 5], omega2, rows);
            if (active) {
                double *ek = ex.ejk + 3 * a.bas[ksh * 8], *el = ex.ejk + 3 * a.bas[lsh * 8];
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    atomic_add(ek + d, gk[d]);
                    atomic_add(el + d, -(gi[d] + gj[d] + gk[d]));
                    gij[d] += gi[d];
                    gij[3 + d] += gj[d];
                }
            }
            wave_sync();
            const uint32_t rest = (nb + lane < qn) ? queue[nb + lane] : 0u;
            wave_sync();
            if (nb + lane < qn) queue[lane] = rest;
            qn -= nb;
            wave_sync();
        }
        if (flush && qn == 0) break;
    }
    double *ei = ex.ejk + 3 * a.bas[sp.ish * 8], *ej = ex.ejk + 3 * a.bas[sp.jsh * 8];
    wave_reduce_scatter<6>(gij, lane, [&](int n, double v) {
        if (v != 0.) atomic_add(n < 3 ? ei + n : ej + n - 3, v);
    });
    if (lane == 0 && a.n_quartets && nsurv) atomicAdd(a.n_quartets, nsurv);
    if (a.quartet_hash && hsum) atomicAdd(a.quartet_hash, hsum);
}

template <int I, int J, int K, int L>
static const void *ip1_lane_fn()
{
    if constexpr (Ip1Lane<I, J, K, L>::ON) return (const void *)jk_ip1_lane_kernel<I, J, K, L>;
    else return nullptr;
}

#define JK_CASE(I, J, K, L) \
    case ((I)*125 + (J)*25 + (K)*5 + (L)): return ip1_lane_fn<I, J, K, L>();
#define JK_CASE_TYPE const void *
#include "jk_dispatch.inc"

const void *jk_ip1_lane_kernel_of(int key)
{
    return dispatch_class(key);
}
