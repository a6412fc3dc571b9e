// Generic Rys kernels: the angular momenta are runtime values, so one kernel
// covers every class up to l = GEN_LMAX (g and h shells) and the first
// derivatives of the ERIs.  They serve the classes the templated per-lane and
// team kernels do not instantiate (any shell with l >= 4) and the per-atom
// energy gradient (no counterpart among the templated kernels).
//
// A workgroup of GEN_TB threads works on one item: an ij pair, a short chunk
// of its kl list and a slice of the rows (i, j) of the Cartesian block (as many
// rows as keep the slice within GEN_ELEMS elements).  Basis sets with g and h
// shells have few of them, so the items are cut small: with one wavefront per
// 256 candidates and the whole block per wavefront, one water molecule
// (def2-TZVP with a g shell on each atom) ran 3-12 wavefronts per launch, up to
// 146 ms for the (gg|gg) class, 357 ms per build; 9.2 ms now.
// The first wavefront applies the survival predicate to the chunk; every
// queued quartet is then evaluated by the whole workgroup, a batch of
// (primitive quartet, root) combinations at a time:
//   * a lane per combination and direction evaluates the root (Chebyshev
//     tables, long-range attenuation as in the templated kernels) and the
//     VRR in i and TRR in k, two rows in registers, into its 2D table in LDS
//     at g[a + c SK];
//   * the bra HRR (independent for every c) and the ket HRR (independent for
//     every (i, j)) are spread over all lanes, a row in registers, in place
//     (strides SJ and SL), so that a table needs exactly
//     (LI+1)(LJ+1)(LK+1)(LL+1) doubles;
//   * every lane owns up to GEN_CH elements of the slice and accumulates their
//     triple products (JK) or their derivative integrals contracted with the
//     two-particle density (gradient); slices below GEN_TB elements are
//     repeated over the lanes, each copy taking its share of the combinations.
// Digestion (JK): the slice and the quartet's density blocks in LDS, one FP64
// atomic per element of the six J/K blocks (symmetry factors of
// rys_contract_jk.cu:156-158,214-220).
// Gradient: the derivative sums of centre k and of centre l (minus the sum of
// the others, by translational invariance) are reduced across the wavefront
// per quartet, those of i and j once per item.
#include "jk_class_kernels.h"
#include "jk_launch.h"

#define GEN_LMAX        5
#define GEN_CH          8
#define GEN_ELEMS       (GEN_TB * GEN_CH)
// work items per launch that the kl chunk aims at
#define GEN_ITEMS       4096
// doubles of LDS for the 2D tables of one batch (a single larger table is
// allowed: 3 tables of the (hh|hh) gradient need 6174)
#define GEN_TAB         4096
// l_i + l_j of the 2D tables (h shells, one more unit on both for gradients)
#define GEN_LPAIR       (2 * GEN_LMAX + 2)

// Cartesian powers of component c of a shell of angular momentum l
// (order lx = l..0, then ly = l - lx..0).
__device__ __forceinline__ void cart_powers(int l, int c, int &x, int &y, int &z)
{
    int lx = l, start = 0;
    while (start + (l - lx + 1) <= c) { start += l - lx + 1; --lx; }
    x = lx;
    y = (l - lx) - (c - start);
    z = l - x - y;
}

// Root i of the N-point Rys rule at x (Chebyshev tables or the large-x
// limit); with omega2 > 0 the rule of the attenuated operator erf(omega r)/r:
// roots and weights of x' = x a, a = omega^2 / (omega^2 + theta), scaled by
// a and sqrt(a).
__device__ void gen_root(const JKRysTable &tab, int N, double x, double theta, double omega2,
                         int i, double &r, double &w)
{
    double sa = 1., aw = 1.;
    if (omega2 > 0.) {
        aw = omega2 / (omega2 + theta);
        sa = sqrt(aw);
        x *= aw;
    }
    if (x >= tab.xmax[N-1]) {
        const double ix = 1. / x;
        r = tab.coef[tab.large_r + N * (N - 1) / 2 + i] * ix;
        w = tab.coef[tab.large_w + N * (N - 1) / 2 + i] * sqrt(ix);
    } else {
        const int D1 = tab.degree + 1;
        const int k = (int)x;
        const double u = 2. * (x - k) - 1., u2 = 2. * u;
        const double *c = tab.coef + tab.off[N-1] + ((int64_t)k * (2 * N) + 2 * i) * D1;
        double r1 = 0., r2 = 0., w1 = 0., w2 = 0.;
        for (int j = D1 - 1; j > 0; --j) {
            double t = fma(u2, r1, c[j] - r2);
            r2 = r1; r1 = t;
            double s = fma(u2, w1, c[D1 + j] - w2);
            w2 = w1; w1 = s;
        }
        r = fma(u, r1, c[0] - r2);
        w = fma(u, w1, c[D1] - w2);
    }
    r *= aw;
    w *= sa;
}

// VRR in a (c = 0) and TRR in c of one root and direction: G(a, c) at
// g[a + c SK], a <= LIJ, c <= LKL.
__device__ __forceinline__ void gen_vrr(double *g, int LIJ, int LKL, int SK, double g00,
                                        double c0, double cp, double b10, double b01,
                                        double b00)
{
    double cur[GEN_LPAIR + 1], prev[GEN_LPAIR + 1];
#pragma unroll
    for (int a = 0; a <= GEN_LPAIR; ++a) { cur[a] = 0.; prev[a] = 0.; }
    cur[0] = g00;
    cur[1] = c0 * g00;
#pragma unroll
    for (int a = 1; a < GEN_LPAIR; ++a)
        if (a < LIJ) cur[a + 1] = c0 * cur[a] + (a * b10) * cur[a - 1];
#pragma unroll
    for (int a = 0; a <= GEN_LPAIR; ++a)
        if (a <= LIJ) g[a] = cur[a];
    for (int c = 0; c < LKL; ++c) {
        double *gn = g + (c + 1) * SK;
        double below = 0.;      // G(a - 1, c)
#pragma unroll
        for (int a = 0; a <= GEN_LPAIR; ++a) {
            if (a > LIJ) continue;
            const double v = cp * cur[a] + (c * b01) * prev[a] + (a * b00) * below;
            prev[a] = below = cur[a];
            cur[a] = v;
            gn[a] = v;
        }
    }
}

// HRR of one line of a table, in place: h[x s0], x <= LA + LB, is combined into
// h[x s0 + y s1], x <= LA, y <= LB (bra: s0 = 1, s1 = SJ; ket: SK, SL).
__device__ __forceinline__ void gen_hrr(double *h, int LA, int LB, int s0, int s1, double r)
{
    double v[GEN_LPAIR + 1];
#pragma unroll
    for (int x = 0; x <= GEN_LPAIR; ++x) v[x] = x <= LA + LB ? h[x * s0] : 0.;
    for (int y = 1; y <= LB; ++y) {
#pragma unroll
        for (int x = 0; x < GEN_LPAIR; ++x) v[x] = v[x + 1] - r * v[x];
#pragma unroll
        for (int x = 0; x <= GEN_LPAIR; ++x)
            if (x <= LA) h[x * s0 + y * s1] = v[x];
    }
}

// Shape of one class: table strides, roots, row slices, batch size.
struct GenShape {
    int LI, LJ, LK, LL;             // of the tables
    int SJ, SK, SL, GS, N;
    int nfk, nfl, nrows, nfkl;
    int rs, nslice;                 // rows per slice, slices
    int lds;                        // doubles
};

__host__ __device__ inline GenShape gen_shape(int li, int lj, int lk, int ll, int mode)
{
    GenShape s;
    // one more unit of angular momentum on i, j, k for derivatives
    const int dd = mode == GEN_IP1 ? 1 : 0;
    s.LI = li + dd; s.LJ = lj + dd; s.LK = lk + dd; s.LL = ll;
    s.SJ = s.LI + 1; s.SK = s.SJ * (s.LJ + 1); s.SL = s.SK * (s.LK + 1);
    s.GS = s.SL * (s.LL + 1);
    s.N = (li + lj + lk + ll + dd) / 2 + 1;
    const int nfi = ncart(li), nfj = ncart(lj);
    s.nfk = ncart(lk); s.nfl = ncart(ll);
    s.nrows = nfi * nfj; s.nfkl = s.nfk * s.nfl;
    s.rs = GEN_ELEMS / s.nfkl < s.nrows ? GEN_ELEMS / s.nfkl : s.nrows;
    s.nslice = (s.nrows + s.rs - 1) / s.rs;
    s.lds = 3 * s.GS > GEN_TAB ? 3 * s.GS : GEN_TAB;
    // digestion: the slice, then D_kl, the rows i and j over the k and l
    // columns, and D_ij
    const int dig = s.rs * s.nfkl + s.nfkl + (nfi + nfj) * (s.nfk + s.nfl) + s.nrows;
    if (mode == GEN_JK && dig > s.lds) s.lds = dig;
    return s;
}

template <int MODE>
__global__ __launch_bounds__(GEN_TB)
void jk_generic_kernel(JKBuildArgs a, TaskBatch batch, GenExtra ex)
{
    __shared__ uint32_t queue[WAVE];
    __shared__ int queue_n;
    __shared__ double meta[GEN_TB];             // gradient: 2 a_i, 2 a_j, 2 a_k per combination
    extern __shared__ double tab[];
    int kl_chunk, unused;
    const int item = select_task(a, batch, kl_chunk, unused);
    const int li = a.li, lj = a.lj, lk = a.lk, ll = a.ll;
    const int tid = threadIdx.x, lane = tid & (WAVE - 1);
    const int nbas = a.nbas, nao = a.nao;
    const size_t nao2 = (size_t)nao * nao;
    select_replica(a);
    if (MODE == GEN_IP1 && a.n_repl > 1)
        ex.ejk += (int64_t)(blockIdx.x % a.n_repl) * a.repl_stride;
    const GenShape s = gen_shape(li, lj, lk, ll, MODE);
    const int slice = item % s.nslice;
    const WorkItem wi = work_item(item / s.nslice, a.npairs_kl, kl_chunk);
    const uint32_t bas_ij = a.pairs_ij[wi.pij];
    const float q_ij = a.q_ij[wi.pij];
    const float kl_cutoff = a.cutoff - q_ij;
    const float penalty = MODE == GEN_JK ? a.dm_penalty : 0.f;
    if (a.q_kl[wi.kl0] + penalty + Q_COND_MARGIN < kl_cutoff) return;
    const bool do_j = MODE == GEN_IP1 ? ex.jf != 0. : a.vj != nullptr;
    const bool do_k = MODE == GEN_IP1 ? ex.kf != 0. : a.vk != nullptr;
    ShellPair sp;
    load_shell_pair(sp, bas_ij, nbas, a.bas, a.env, a.ao_loc);
    // survivors of the chunk (at most one wavefront of candidates)
    if (tid < WAVE) {
        const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
        const int pkl = wi.kl0 + lane;
        bool keep = false;
        if (pkl < wi.kl1) {
            const float q_kl = a.q_kl[pkl];
            const uint32_t bkl = a.pairs_kl[pkl];
            if (MODE == GEN_JK)
                keep = survives(q_kl, kl_cutoff, a.dm_penalty, bas_ij, bkl, sp.ish, sp.jsh, nbas,
                                a.dm_cond, a.screen, a.swap_ijkl != 0, q_ij, a.cutoff);
            else
                keep = survives_ejk(q_kl, kl_cutoff, bas_ij, bkl, sp.ish, sp.jsh, nbas,
                                    a.dm_cond, do_j, do_k);
            if (a.quartet_hash && keep && slice == 0)
                atomicAdd(a.quartet_hash, task_mix(a, bas_ij, bkl));
        }
        const uint64_t m = __ballot(keep);
        if (keep) queue[__popcll(m & lt_mask)] = pkl;
        if (lane == 0) {
            queue_n = __popcll(m);
            if (a.n_quartets && slice == 0 && m)
                atomicAdd(a.n_quartets, (unsigned long long)__popcll(m));
        }
    }
    __syncthreads();
    const int qn = queue_n;
    if (qn == 0) return;

    const int nfj = ncart(lj), nfi = ncart(li);
    const int r0 = slice * s.rs, r1 = min(r0 + s.rs, s.nrows);
    const int ne = (r1 - r0) * s.nfkl;          // elements of the slice
    // copies of a slice below GEN_TB elements: copy `sub` of nsub
    int ep = GEN_TB;
    while (ep / 2 >= ne) ep >>= 1;
    const int nsub = GEN_TB / ep, sub = tid / ep, e_first = tid & (ep - 1);
    // the lane's elements: table offsets and Cartesian powers
    int ox[GEN_CH], oy[GEN_CH], oz[GEN_CH];
    uint32_t pw[GEN_CH];
#pragma unroll
    for (int c = 0; c < GEN_CH; ++c) {
        const int e = e_first + c * GEN_TB;
        ox[c] = oy[c] = oz[c] = 0;
        pw[c] = 0;
        if (e >= ne) continue;
        const int row = r0 + e / s.nfkl, kl = e % s.nfkl;
        int ix, iy, iz, jx, jy, jz, kx, ky, kz, lx, ly, lz;
        cart_powers(li, row / nfj, ix, iy, iz);
        cart_powers(lj, row % nfj, jx, jy, jz);
        cart_powers(lk, kl / s.nfl, kx, ky, kz);
        cart_powers(ll, kl % s.nfl, lx, ly, lz);
        ox[c] = ix + jx * s.SJ + kx * s.SK + lx * s.SL;
        oy[c] = iy + jy * s.SJ + ky * s.SK + ly * s.SL;
        oz[c] = iz + jz * s.SJ + kz * s.SK + lz * s.SL;
        // powers packed 4 bits each: ix iy iz jx jy jz kx ky (kz = lk - kx - ky)
        pw[c] = ix | iy << 4 | iz << 8 | jx << 12 | jy << 16 | jz << 20 | kx << 24 | ky << 28;
    }
    const double omega2 = a.omega * a.omega;
    const int nij = a.iprim * a.jprim, nkl = a.kprim * a.lprim;
    const int ncomb = nij * nkl * s.N;
    const double *pdij = a.pdata_ij + (size_t)wi.pij * nij * PREC;
    const int i0 = sp.i0, j0 = sp.j0;
    const int LIJ = s.LI + s.LJ, LKL = s.LK + s.LL;
    int cb = s.lds / (3 * s.GS);
    cb = min(min(cb, GEN_TB / 3), ncomb);
    double gij[6];
#pragma unroll
    for (int t = 0; t < 6; ++t) gij[t] = 0.;

    for (int q = 0; q < qn; ++q) {
        const int pkl = queue[q];
        const uint32_t bas_kl = a.pairs_kl[pkl];
        const int ksh = bas_kl / nbas, lsh = bas_kl - (bas_kl / nbas) * nbas;
        double fac_sym = a.scale;
        if (sp.ish == sp.jsh) fac_sym *= .5;
        if (ksh == lsh) fac_sym *= .5;
        if (bas_ij == bas_kl) fac_sym *= .5;
        const double *rk = a.env + a.bas[ksh * 8 + 7], *rl = a.env + a.bas[lsh * 8 + 7];
        const double rk3[3] = {rk[0], rk[1], rk[2]};
        const double rkl[3] = {rl[0] - rk[0], rl[1] - rk[1], rl[2] - rk[2]};
        const int k0 = a.ao_loc[ksh], l0 = a.ao_loc[lsh];
        const double *pdkl = a.pdata_kl + (size_t)pkl * nkl * PREC;
        double acc[GEN_CH];
#pragma unroll
        for (int c = 0; c < GEN_CH; ++c) acc[c] = 0.;
        if (MODE == GEN_IP1) {
            // two-particle density of the elements (rys_contract_jk_ip1.cu:523-577)
#pragma unroll
            for (int c = 0; c < GEN_CH; ++c) {
                const int e = e_first + c * GEN_TB;
                if (e >= ne) continue;
                const int row = r0 + e / s.nfkl, kl = e % s.nfkl;
                const size_t I = i0 + row / nfj, J = j0 + row % nfj;
                const size_t K = k0 + kl / s.nfl, L = l0 + kl % s.nfl;
                const double *D = a.dm;
                double g2 = 0., dji = 0., dlk = 0.;
                for (int id = 0; id < a.n_dm; ++id, D += nao2) {
                    if (do_k) g2 += ex.kf * (D[J*nao+K] * D[L*nao+I] + D[J*nao+L] * D[K*nao+I]);
                    dji += D[J*nao+I]; dlk += D[L*nao+K];
                }
                acc[c] = (g2 + ex.jf * dji * dlk) * fac_sym;    // the element's weight
            }
        }
        double gsum[9];
#pragma unroll
        for (int t = 0; t < 9; ++t) gsum[t] = 0.;
        for (int c0 = 0; c0 < ncomb; c0 += cb) {
            const int nc = min(cb, ncomb - c0);
            __syncthreads();        // the previous batch or digestion has read the tables
            if (tid < 3 * nc) {
                const int c = tid / 3, d = tid - 3 * c;
                const int pq = (c0 + c) / s.N, r = c0 + c - pq * s.N;
                const int kp = pq / nij, ip = pq - kp * nij;
                const double *qr = pdkl + kp * PREC, *pr = pdij + ip * PREC;
                const double akl = qr[0], aij = pr[0];
                const double x = pr[2] - qr[2], y = pr[3] - qr[3], z = pr[4] - qr[4];
                const double rr = x * x + y * y + z * z;
                const double r_aa = 1. / (aij + akl);
                const double theta = aij * akl * r_aa;
                double rt, wt;
                gen_root(a.rys, s.N, theta * rr, theta, omega2, r, rt, wt);
                const double rt_aa = rt * r_aa;
                const double rt_aij = rt_aa * akl, rt_akl = rt_aa * aij;
                const double pqd = d == 0 ? x : d == 1 ? y : z;
                const double rid = d == 0 ? sp.ri[0] : d == 1 ? sp.ri[1] : sp.ri[2];
                const double rkd = d == 0 ? rk3[0] : d == 1 ? rk3[1] : rk3[2];
                const double g00 = d == 2 ? wt * pr[5] * qr[5] * sqrt(r_aa) *
                                            (MODE == GEN_JK ? fac_sym : 1.) : 1.;
                gen_vrr(tab + tid * s.GS, LIJ, LKL, s.SK, g00,
                        pr[2 + d] - rid - rt_aij * pqd, qr[2 + d] - rkd + rt_akl * pqd,
                        .5 * pr[1] * (1. - rt_aij), .5 * qr[1] * (1. - rt_akl), .5 * rt_aa);
                if (MODE == GEN_IP1 && d == 0) {
                    meta[3 * c] = 2. * a.env[sp.pexpi + ip / a.jprim];
                    meta[3 * c + 1] = 2. * a.env[sp.pexpj + ip % a.jprim];
                    meta[3 * c + 2] = 2. * a.env[a.bas[ksh * 8 + 5] + kp / a.lprim];
                }
            }
            __syncthreads();
            if (s.LJ > 0) {
                for (int n = tid; n < 3 * nc * (LKL + 1); n += GEN_TB) {
                    const int t = n / (LKL + 1), c = n - t * (LKL + 1);
                    const int d = t % 3;
                    gen_hrr(tab + t * s.GS + c * s.SK, s.LI, s.LJ, 1, s.SJ,
                            d == 0 ? sp.rij[0] : d == 1 ? sp.rij[1] : sp.rij[2]);
                }
                __syncthreads();
            }
            if (s.LL > 0) {
                for (int n = tid; n < 3 * nc * s.SK; n += GEN_TB) {
                    const int t = n / s.SK, ij = n - t * s.SK;
                    const int d = t % 3;
                    gen_hrr(tab + t * s.GS + ij, s.LK, s.LL, s.SK, s.SL,
                            d == 0 ? rkl[0] : d == 1 ? rkl[1] : rkl[2]);
                }
                __syncthreads();
            }
            for (int cc = sub; cc < nc; cc += nsub) {
                const double *gx = tab + 3 * cc * s.GS;
                const double *gy = gx + s.GS, *gz = gy + s.GS;
                double ai2 = 0., aj2 = 0., ak2 = 0.;
                if (MODE == GEN_IP1) { ai2 = meta[3*cc]; aj2 = meta[3*cc+1]; ak2 = meta[3*cc+2]; }
#pragma unroll
                for (int c = 0; c < GEN_CH; ++c) {
                    if (e_first + c * GEN_TB >= ne) continue;
                    const double x = gx[ox[c]], y = gy[oy[c]], z = gz[oz[c]];
                    if (MODE == GEN_JK) {
                        acc[c] = fma(x * y, z, acc[c]);
                    } else {
                        const uint32_t p = pw[c];
                        const int ix = p & 15, iy = p >> 4 & 15, iz = p >> 8 & 15;
                        const int jx = p >> 12 & 15, jy = p >> 16 & 15, jz = p >> 20 & 15;
                        const int kx = p >> 24 & 15, ky = p >> 28, kz = lk - kx - ky;
                        const double w = acc[c];
                        // d/dA: 2 ai g(i+1) - i g(i-1), likewise B (j), C (k)
                        const double dxi = ai2 * gx[ox[c] + 1] - (ix ? ix * gx[ox[c] - 1] : 0.);
                        const double dyi = ai2 * gy[oy[c] + 1] - (iy ? iy * gy[oy[c] - 1] : 0.);
                        const double dzi = ai2 * gz[oz[c] + 1] - (iz ? iz * gz[oz[c] - 1] : 0.);
                        const double dxj = aj2 * gx[ox[c] + s.SJ] - (jx ? jx * gx[ox[c] - s.SJ] : 0.);
                        const double dyj = aj2 * gy[oy[c] + s.SJ] - (jy ? jy * gy[oy[c] - s.SJ] : 0.);
                        const double dzj = aj2 * gz[oz[c] + s.SJ] - (jz ? jz * gz[oz[c] - s.SJ] : 0.);
                        const double dxk = ak2 * gx[ox[c] + s.SK] - (kx ? kx * gx[ox[c] - s.SK] : 0.);
                        const double dyk = ak2 * gy[oy[c] + s.SK] - (ky ? ky * gy[oy[c] - s.SK] : 0.);
                        const double dzk = ak2 * gz[oz[c] + s.SK] - (kz ? kz * gz[oz[c] - s.SK] : 0.);
                        const double yz = w * (y * z), xz = w * (x * z), xy = w * (x * y);
                        gsum[0] = fma(dxi, yz, gsum[0]);
                        gsum[1] = fma(dyi, xz, gsum[1]);
                        gsum[2] = fma(dzi, xy, gsum[2]);
                        gsum[3] = fma(dxj, yz, gsum[3]);
                        gsum[4] = fma(dyj, xz, gsum[4]);
                        gsum[5] = fma(dzj, xy, gsum[5]);
                        gsum[6] = fma(dxk, yz, gsum[6]);
                        gsum[7] = fma(dyk, xz, gsum[7]);
                        gsum[8] = fma(dzk, xy, gsum[8]);
                    }
                }
            }
        }
        if (MODE == GEN_IP1) {
            double kl[6];
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                kl[t] = gsum[6 + t];
                kl[3 + t] = -(gsum[t] + gsum[3 + t] + gsum[6 + t]);
                gij[t] += gsum[t];
                gij[3 + t] += gsum[3 + t];
            }
            const int ka = a.bas[ksh * 8], la = a.bas[lsh * 8];
            wave_reduce_scatter<6>(kl, lane, [&](int n, double v) {
                if (v != 0.) atomic_add(ex.ejk + (n < 3 ? ka * 3 + n : la * 3 + n - 3), v);
            });
            continue;
        }
        // ---- digestion of the slice
        double *stage = tab;
        const int dw = s.nfk + s.nfl;
        double *dkl = stage + (r1 - r0) * s.nfkl, *drow = dkl + s.nfkl;
        double *dij = drow + (nfi + nfj) * dw;
        __syncthreads();
        if (sub == 0) {
#pragma unroll
            for (int c = 0; c < GEN_CH; ++c)
                if (e_first + c * GEN_TB < ne) stage[e_first + c * GEN_TB] = acc[c];
        }
        __syncthreads();
        if (sub > 0 && e_first < ne) lds_add(stage + e_first, acc[0]);
        for (int id = 0; id < a.n_dm; ++id) {
            const double *D = a.dm + id * nao2;
            __syncthreads();
            for (int n = tid; n < s.nfkl; n += GEN_TB)
                dkl[n] = D[(size_t)(k0 + n / s.nfl) * nao + l0 + n % s.nfl];
            for (int n = tid; n < (nfi + nfj) * dw; n += GEN_TB) {
                const int r = n / dw, c = n - r * dw;
                const size_t ao = r < nfi ? i0 + r : j0 + r - nfi;
                drow[n] = D[ao * nao + (c < s.nfk ? k0 + c : l0 + c - s.nfk)];
            }
            for (int n = tid; n < s.nrows; n += GEN_TB)
                dij[n] = D[(size_t)(i0 + n / nfj) * nao + j0 + n % nfj];
            __syncthreads();
            if (do_j) {
                double *J = a.vj + id * nao2;
                for (int n = tid; n < s.nfkl; n += GEN_TB) {
                    double v = 0.;
                    for (int r = r0; r < r1; ++r)
                        v = fma(stage[(r - r0) * s.nfkl + n], dij[r], v);
                    atomic_add(J + (size_t)(k0 + n / s.nfl) * nao + l0 + n % s.nfl, v);
                }
                // 16 lanes per row
                for (int r = r0 + tid / 16; r < r1; r += GEN_TB / 16) {
                    double v = 0.;
                    for (int n = tid & 15; n < s.nfkl; n += 16)
                        v = fma(stage[(r - r0) * s.nfkl + n], dkl[n], v);
#pragma unroll
                    for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 16);
                    if ((tid & 15) == 0)
                        atomic_add(J + (size_t)(i0 + r / nfj) * nao + j0 + r % nfj, v);
                }
            }
            if (do_k) {
                double *K = a.vk + id * nao2;
                const int ilo = r0 / nfj, ihi = (r1 - 1) / nfj;
                const int ni = ihi - ilo + 1;
                // K_ik (D_jl), K_il (D_jk), then K_jk (D_il), K_jl (D_ik)
                for (int n = tid; n < (ni + nfj) * dw; n += GEN_TB) {
                    const int x = n / dw, m = n - x * dw;
                    const bool bra_i = x < ni;
                    double v = 0.;
                    // partner index y of the row: j for x = i, i for x = j
                    const int y0 = bra_i ? 0 : ilo, y1 = bra_i ? nfj : ihi + 1;
                    for (int y = y0; y < y1; ++y) {
                        const int r = bra_i ? (ilo + x) * nfj + y : y * nfj + x - ni;
                        if (r < r0 || r >= r1) continue;
                        const double *srow = stage + (r - r0) * s.nfkl;
                        const double *dr = drow + (bra_i ? nfi + y : y) * dw;
                        if (m < s.nfk) {
                            for (int l = 0; l < s.nfl; ++l)
                                v = fma(srow[m * s.nfl + l], dr[s.nfk + l], v);
                        } else {
                            for (int k = 0; k < s.nfk; ++k)
                                v = fma(srow[k * s.nfl + m - s.nfk], dr[k], v);
                        }
                    }
                    const size_t row = bra_i ? i0 + ilo + x : j0 + x - ni;
                    atomic_add(K + row * nao + (m < s.nfk ? k0 + m : l0 + m - s.nfk), v);
                }
            }
        }
    }
    if (MODE == GEN_IP1) {
        const int ia = a.bas[sp.ish * 8], ja = a.bas[sp.jsh * 8];
        wave_reduce_scatter<6>(gij, lane, [&](int n, double v) {
            if (v != 0.) atomic_add(ex.ejk + (n < 3 ? ia * 3 + n : ja * 3 + n - 3), v);
        });
    }
}

// Candidates per work item and workgroups of one task; dynamic LDS in bytes.
bool jk_generic_plan(const JKTask &k, int mode, TaskDesc &d, long &blocks, size_t &lds)
{
    if (k.li > GEN_LMAX || k.lj > GEN_LMAX || k.lk > GEN_LMAX || k.ll > GEN_LMAX) return false;
    const GenShape s = gen_shape(k.li, k.lj, k.lk, k.ll, mode);
    lds = sizeof(double) * s.lds;
    // the chunk that leaves GEN_ITEMS items, at most one wavefront of candidates
    const double all = (double)k.npairs_ij * k.npairs_kl * s.nslice;
    int chunk = all / GEN_ITEMS < WAVE ? (int)(all / GEN_ITEMS) : WAVE;
    if (chunk < 1) chunk = 1;
    d.kl_chunk = chunk;
    blocks = (long)k.npairs_ij * ((k.npairs_kl + chunk - 1) / chunk) * s.nslice;
    return true;
}

const void *jk_generic_kernel_of(int mode)
{
    return mode == GEN_JK ? (const void *)jk_generic_kernel<GEN_JK>
                          : (const void *)jk_generic_kernel<GEN_IP1>;
}
