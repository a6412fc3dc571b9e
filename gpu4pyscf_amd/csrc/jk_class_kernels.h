// Device code of the class kernels (per-lane and team kernels) and the class
// information for their launches (jk_launch.hip), shared by the translation units
// that instantiate the angular classes (jk_classes.hip, compiled once per part).
// Direct-SCF J/K kernels for MI355X (gfx950), FP64 Rys quadrature.
//
// One launch evaluates one angular class (li,lj,lk,ll) of screened shell
// quartets and contracts it with the density matrices into J and K.
//
// Work decomposition: a work item is (one ij shell pair, one chunk of the kl
// pair list, or one kl column window of it).  The block scans the kl
// candidates of its chunk, applies the survival predicate of
// gpu4pyscf/lib/gvhf-rys/create_tasks.cu:114-180 and compacts the survivors
// into an LDS queue with wavefront ballots; queued quartets are then
// evaluated
//   * by the per-lane kernel (small classes, and some d/f classes in chunks of
//     block rows): one quartet per lane, the 2D Rys integrals and the
//     Cartesian block (or a chunk of its rows) in VGPRs;
//   * by the team kernel (large classes): a team of lanes per quartet, the
//     2D integrals of all roots staged in LDS, each lane owning one (i,j) row
//     of the block, the block staged through LDS for the contraction.
// A launch may run its task with bra and ket exchanged (swap_ijkl); the
// survival test and checksum then follow the task's own order.
// Digestion follows gpu4pyscf/lib/gvhf-rys/rys_contract_jk.cu:291-330 (four K
// blocks and two J blocks per quartet, symmetry factors of :156-158,214-220).
// On this 8-XCD part an FP64 atomic add into HBM is resolved on the memory
// side, so the kernels reduce in registers and LDS first: J_ij (common to a
// work item) across the wavefront or in the row-owning lane, the K rows of
// the work item's i and j AOs in LDS (per-lane kernel), the density blocks
// read by the digestion staged in LDS; what remains per quartet (J_kl, and
// K in the team kernel) goes to HBM with FP64 atomics.
// Rys roots: for up to three roots the Gauss rule of Boys moments taken from
// Taylor series of one of them; otherwise Chebyshev tables; both generated
// by gen_rys_table.py.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>
#include <type_traits>
#include <atomic>
#include "../../include/jkhip.h"

#define PI_FAC          34.98683665524972497    // 2 pi^(5/2)
#define Q_COND_MARGIN   4.f
#define WAVE            64
#define RYS_DEG_MAX     15
// classes whose Cartesian block plus three 2D tables fit in LANE_MAX
// doubles run one quartet per lane, the others on teams of lanes.
// Measured (ms per 32-water def2-TZVP build): 120 -> 720, 150 -> 679,
// 170 -> 660 (adds the (dd|ps)-sized classes), 240 -> 682; 64-water
// def2-TZVP build: 95 -> 3261, 120 -> 3271, 170 -> 3134.
#ifndef LANE_MAX
#define LANE_MAX        170
#endif
// classes whose block does not fit LANE_MAX with its 2D tables run per lane
// in chunks of rows i when listed in LaneChunked (below), or when they need
// at most LANE_MAX_CHUNKS chunks (1: the list only); the others on teams
#ifndef LANE_MAX_CHUNKS
#define LANE_MAX_CHUNKS 1
#endif
// doubles of one chunk (its rows of the block plus three 2D tables).  220
// with up to 3 chunks: (fp|pp) 69.9 -> 60.7 ms and (ff|ps) 55.5 -> 50.5 ms on
// the 64-water build, every class chunked before slower (larger chunks spill)
#ifndef LANE_CHUNK_MAX
#define LANE_CHUNK_MAX  LANE_MAX
#endif
// a block size the per-lane kernel leaves to the team kernel (0: none);
// sending the spilling (ff|ss)/(fs|fs) (100) or (dd|ps)-sized (108) classes
// back to the team kernel measured 658 and 670 ms against 652
#ifndef LANE_SKIP_NF
#define LANE_SKIP_NF    0
#endif
// launch shapes: work items of the per-lane kernel target LANE_ITEMS blocks
// per launch with at least LANE_MIN_CHUNK kl candidates each; the team
// kernel scans TEAM_KL_CHUNK candidates per work item.  Measured on the
// 32-water def2-TZVP build (ms per build): team chunk 256/128/64/48/32 ->
// 1280/1143/1109/1065/1077 with 2048 lane items; lane items 4096 -> 2048
// at team chunk 256: 1280 -> 1236; without team K rows, lane items
// 2048 -> 1024: 883 -> 873.
#ifndef LANE_ITEMS
#define LANE_ITEMS      1024
#endif
#ifndef LANE_MIN_CHUNK
#define LANE_MIN_CHUNK  256
#endif
#ifndef TEAM_KL_CHUNK
#define TEAM_KL_CHUNK   48
#endif
// LDS K rows of the team kernel (0 none, 1 K_il/K_jl) and its minimum
// waves per SIMD (register budget).  With short work items zeroing and
// flushing the rows costs more than the atomics they save: 1065 -> 884 ms
// per build without them; a minimum of 2 or 3 waves per SIMD (fewer
// registers) measured 1105 and 1197 ms.
#ifndef TEAM_KROWS
#define TEAM_KROWS      0
#endif
// team kernel over kl column windows (kl_win[1]) with all four K blocks in
// LDS, for launches of at least TEAM_KWIN_MIN_ITEMS (ij pair, window) items.
// Off (used only under kl_win_policy 1): the rows cost more workgroups per
// CU than the atomics they save.  64-water def2-TZVP build, team kernels on
// one stream: 1080 ms without; with windows of 64 / 96 / 128 AOs 1159 /
// 1406 / 1512 ms (32-water: 280 without, 325 with 64-AO windows).
#ifndef TEAM_KWIN
#define TEAM_KWIN       0
#endif
// smallest workgroup of the team kernel (threads; 64, 128 or 256).  64-water
// def2-TZVP build, team kernels on one stream: 1082 ms with 64; 256: 1264 ms,
// 1199-1210 ms with K rows over 96- or 128-AO kl windows; 128 with 96-AO
// windows: 1176 ms.
#ifndef TEAM_TB_MIN
#define TEAM_TB_MIN     64
#endif
#ifndef TEAM_KWIN_MIN_ITEMS
#define TEAM_KWIN_MIN_ITEMS 2048
#endif
#ifndef TEAM_MIN_WAVES
#define TEAM_MIN_WAVES  1
#endif
// team kernel: evaluate several primitive quartets of a quartet per pass
// (roots, 2D tables and triple products of PB primitive quartets between
// three block barriers) instead of one.  Off: the larger LDS footprint cost
// more than the barriers it saves (64-water def2-TZVP build, team kernels on
// one stream: 1082 ms without, 1122 ms with)
#ifndef TEAM_PRIM_BATCH
#define TEAM_PRIM_BATCH 0
#endif
// LDS rows of the per-lane kernel: 2 = K_ik/K_jk and K_il/K_jl, 1 = K_il/K_jl
// only; LANE_DROWS also stages the density rows (883 ms per build; 1061
// with K_il/K_jl rows only, 887 without the density rows)
#ifndef LANE_KROWS
#define LANE_KROWS      2
#endif
#ifndef LANE_DROWS
#define LANE_DROWS      1
#endif
// K_ik / K_jk LDS rows of the per-lane kernel: 1 = the lanes of a run of
// equal k shell first sum their values across the wavefront and the run's
// last lane adds once (no same-address LDS atomics within the run), 0 = every
// lane adds its own values.  Measured on the 64-water def2-TZVP build: 3130 ms
// with 0, 3229 ms with 1 (LDS bank conflicts are 0.05-1.5 % of the time of
// these kernels; the cross-lane sums cost more than the conflicts they avoid)
#ifndef LANE_KIK_SEGSUM
#define LANE_KIK_SEGSUM 0
#endif

void jk_set_error(const char *msg);

// ---------------------------------------------------------------- helpers
__host__ __device__ constexpr int ncart(int l) { return (l + 1) * (l + 2) / 2; }

template <int L>
struct CartPow {
    int x[ncart(L)], y[ncart(L)], z[ncart(L)];
    constexpr CartPow() : x(), y(), z() {
        int c = 0;
        for (int lx = L; lx >= 0; --lx)
            for (int ly = L - lx; ly >= 0; --ly) {
                x[c] = lx; y[c] = ly; z[c] = L - lx - ly; ++c;
            }
    }
};

__device__ __forceinline__ void atomic_add(double *p, double v)
{
    unsafeAtomicAdd(p, v);
}

// Replicated accumulation (JKBuildArgs.n_repl): this workgroup's copy of
// vj/vk.
__device__ __forceinline__ void select_replica(JKBuildArgs &a)
{
    if (a.n_repl > 1) {
        const int64_t off = (int64_t)(blockIdx.x % a.n_repl) * a.repl_stride;
        if (a.vj) a.vj += off;
        if (a.vk) a.vk += off;
    }
}

// LDS accumulation: workgroup scope, so that it cannot be merged with the
// device-scope HBM atomics of a sibling branch into one generic atomic
__device__ __forceinline__ void lds_add(double *p, double v)
{
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// A double in LDS by its own address space: where a value comes from LDS in one
// branch and from HBM in the other, generic pointers let the compiler merge the
// two loads into a flat one, which is slower than either and completes only
// behind the wavefront's outstanding atomics.
typedef __attribute__((address_space(3))) double lds_double;

__device__ __forceinline__ void lds_add(lds_double *p, double v)
{
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        v += __shfl_xor(v, off, WAVE);
    return v;
}

// Sums M values over the 64 lanes of a wavefront and hands each total to
// one lane (reduce-scatter by recursive halving): at the step with lane bit
// b, lanes with bit b set keep the upper half of their values and add the
// partner's upper half, the others the lower half.  About M shuffles instead
// of 6 M for M separate butterfly sums.  v holds the M values of this lane
// and is overwritten; `put(n, x)` is called for every n < M, on the lane
// that holds the total x of value n.
// Value of the partner lane at the reduce-scatter step of lane bit BIT.
// Steps inside a 16-lane row use DPP moves (no LDS crossbar): lane ^ 1 and
// lane ^ 2 by quad permutes, lane ^ 8 by a row rotation of 8, and for
// BIT = 4 the half-row mirror, lane ^ 7: that partner also has the opposite
// bit 2 and the same higher bits, and its lanes summed so far are disjoint
// from this lane's, so the later ^ 2 and ^ 1 steps still cover all eight
// low-bit patterns.  The steps across rows (lane ^ 16, lane ^ 32) use the
// row-swap moves of gfx950: permlane16_swap(x, x) leaves row r ^ 1's values
// in its second result on even rows and in its first on odd rows,
// permlane32_swap(x, x) the other half's in its second result on lanes
// 0-31 and in its first on lanes 32-63.
// 0: LDS crossbar shuffles only; 1: DPP for the in-row steps; 2: also the
// row swaps (64-water build 2017 -> 1998 -> 1989 ms)
#ifndef WAVE_DPP
#define WAVE_DPP 2
#endif
template <int BIT>
__device__ __forceinline__ double partner_value(double x)
{
    constexpr int CTRL = BIT == 1 ? 0xB1 : BIT == 2 ? 0x4E : BIT == 4 ? 0x141 :
                         BIT == 8 ? 0x128 : -1;
    if constexpr (WAVE_DPP && CTRL >= 0) {
        const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xF, 0xF, false);
        const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xF, 0xF, false);
        return __hiloint2double(hi, lo);
    } else if constexpr (WAVE_DPP > 1 && (BIT == 16 || BIT == 32)) {
        const bool up = (__lane_id() & BIT) != 0;
        const int lo = __double2loint(x), hi = __double2hiint(x);
        if constexpr (BIT == 16) {
            const auto a = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
            const auto b = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
            return __hiloint2double(up ? (int)b[0] : (int)b[1], up ? (int)a[0] : (int)a[1]);
        } else {
            const auto a = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
            const auto b = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
            return __hiloint2double(up ? (int)b[0] : (int)b[1], up ? (int)a[0] : (int)a[1]);
        }
    } else {
        return __shfl_xor(x, BIT, WAVE);
    }
}

template <int M, int BIT, typename F>
__device__ __forceinline__ void reduce_scatter_step(double *v, int lane, int base, int nvalid,
                                                    F &put)
{
    if constexpr (BIT == 0) {
#pragma unroll
        for (int t = 0; t < M; ++t)
            if (t < nvalid) put(base + t, v[t]);
    } else {
        constexpr int H = (M + 1) / 2;
        const bool hi = (lane & BIT) != 0;
        double w[H];
#pragma unroll
        for (int t = 0; t < H; ++t) {
            const double lo_v = v[t];
            const double hi_v = (H + t < M) ? v[H + t] : 0.;
            const double mine = hi ? hi_v : lo_v;
            const double send = hi ? lo_v : hi_v;
            w[t] = mine + partner_value<BIT>(send);
        }
        const int nv = hi ? (nvalid > H ? nvalid - H : 0) : (nvalid < H ? nvalid : H);
        reduce_scatter_step<H, BIT / 2>(w, lane, hi ? base + H : base, nv, put);
    }
}

template <int M, typename F>
__device__ __forceinline__ void wave_reduce_scatter(double *v, int lane, F &&put)
{
    reduce_scatter_step<M, WAVE / 2>(v, lane, 0, M, put);
}

// Orders LDS accesses of the lanes of one wavefront (no block barrier).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Inclusive segmented sum over lanes with equal, contiguous segment ids (the
// last lane of a segment receives the segment total), with the segment
// comparisons done once: same[s] says whether lane - 2^s belongs to this
// lane's segment.
struct SegMask { bool same[6]; };

__device__ __forceinline__ SegMask seg_mask(int seg, int lane)
{
    SegMask m;
#pragma unroll
    for (int s = 0; s < 6; ++s) {
        const int off = 1 << s;
        const int o = __shfl_up(seg, off, WAVE);
        m.same[s] = lane >= off && o == seg;
    }
    return m;
}

__device__ __forceinline__ double seg_sum(double v, const SegMask &m)
{
#pragma unroll
    for (int s = 0; s < 6; ++s) {
        const double u = __shfl_up(v, 1 << s, WAVE);
        if (m.same[s]) v += u;
    }
    return v;
}

// Reciprocal, quotient, reciprocal square root and square root of normal
// numbers, within an ulp: the hardware estimates (24 bits) with two Newton
// steps, 5 to 8 instructions where the IEEE forms take 10 to 20.
__device__ __forceinline__ double rcp64(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.), r, r);
    return fma(fma(-x, r, 1.), r, r);
}

__device__ __forceinline__ double div64(double a, double b)
{
    double r = __builtin_amdgcn_rcp(b);
    r = fma(fma(-b, r, 1.), r, r);
    const double q = a * r;
    return fma(fma(-b, q, a), r, q);
}

__device__ __forceinline__ double rsqrt64(double x)
{
    double y = __builtin_amdgcn_rsq(x);
    y = fma(y, fma(-x * y, .5 * y, .5), y);
    return fma(y, fma(-x * y, .5 * y, .5), y);
}

__device__ __forceinline__ double sqrt64(double x)
{
    double y = __builtin_amdgcn_rsq(x);
    y = fma(y, fma(-x * y, .5 * y, .5), y);
    const double s = x * y;
    return fma(fma(-s, s, x), .5 * y, s);
}

// the same for the FP32 quartets
__device__ __forceinline__ float rcp64(float x) { return 1.f / x; }
__device__ __forceinline__ float rsqrt64(float x) { return sqrtf(1.f / x); }

// Moment rows of the N-point rule in LDS (JKRysTable.boys: N = 1, 2, 3), one
// copy per workgroup.  A row is read whole by every lane at an address of its
// own; from the caches such a gather occupies the address units for 64 lines,
// and they were 65 to 80 % busy in the s and p classes ((ss|ss), (ps|ss),
// (ps|ps)).  One Taylor series of the highest moment, one of the exponential
// and a downward recursion replace a series per moment: 27 + 2N fused
// operations against 32 N.  Rows of 14 doubles 0.5 apart keep the copy at 9 to
// 12 KB (a grid of 0.1 for all moments took 56 KB, larger than the L1).
// 48 waters (def2-TZVP): (fs|ps) 45.8 -> 37.2 ms, (fp|ps) 34.7 -> 31.7, (dp|ps)
// 42.9 -> 40.6, the whole build 1019 -> 1000; 8 waters (def2-SVP) 2.91 -> 2.55.
#define MOMENT_TERMS 12
#define MOMENT_STEP .5
__host__ __device__ constexpr int moment_rows(int n) { return n == 1 ? 79 : n == 2 ? 95 : n == 3 ? 109 : 0; }
typedef double double2v __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) double2v lds_double2;

template <int N>
struct MomentRows {
    static constexpr int SIZE = N <= 3 ? moment_rows(N) * JK_BOYS_M : 2;    // doubles
};

// copies the rows (a barrier must follow)
template <int N>
__device__ __forceinline__ void load_moment_rows(double *buf, const JKRysTable &tab, int tid,
                                                 int nthreads)
{
    if constexpr (N <= 3) {
        const int before = (N > 1 ? moment_rows(1) : 0) + (N > 2 ? moment_rows(2) : 0);
        const double2v *src = (const double2v *)(tab.coef + tab.boys + before * JK_BOYS_M);
        lds_double2 *dst = (lds_double2 *)(lds_double *)buf;
        for (int n = tid; n < MomentRows<N>::SIZE / 2; n += nthreads) dst[n] = src[n];
    }
}

// A constant that is put into scalar registers where it is used: left to
// itself the compiler keeps the factorials of the two series in 24 vector
// registers over the whole kernel ((ss|ss) 86 -> 124, (ps|ss) 119 -> 142).
__device__ __forceinline__ double scalar_const(double c)
{
    asm volatile("" : "+s"(c));
    return c;
}

// Boys moments F_0..F_{2N-1}(x), x < xmax[N-1]
template <int N>
__device__ __forceinline__ void boys_moments(const lds_double *rows, double x, double *f)
{
    constexpr int M = 2 * N - 1;
    constexpr double INV_FACT[13] = {1., 1., 1. / 2, 1. / 6, 1. / 24, 1. / 120, 1. / 720,
                                     1. / 5040, 1. / 40320, 1. / 362880, 1. / 3628800,
                                     1. / 39916800, 1. / 479001600};
    int g = (int)fma(x, 1. / MOMENT_STEP, .5);
    g = g < moment_rows(N) - 1 ? g : moment_rows(N) - 1;
    const double d = fma((double)g, MOMENT_STEP, -x);
    const lds_double2 *p = (const lds_double2 *)(rows + g * JK_BOYS_M);
    double c[JK_BOYS_M];
#pragma unroll
    for (int k = 0; k < JK_BOYS_M / 2; ++k) {
        const double2v v = p[k];
        c[2 * k] = v.x; c[2 * k + 1] = v.y;
    }
    double s = c[MOMENT_TERMS - 1], e = scalar_const(INV_FACT[12]);
#pragma unroll
    for (int k = MOMENT_TERMS - 2; k >= 0; --k) s = fma(s, d, c[k]);
#pragma unroll
    for (int k = 11; k >= 0; --k)
        e = fma(e, d, k > 2 ? scalar_const(INV_FACT[k]) : INV_FACT[k]);
    e *= c[MOMENT_TERMS];
    const double x2 = 2. * x;
    f[M] = s;
#pragma unroll
    for (int m = M; m > 0; --m) f[m - 1] = fma(x2, f[m], e) * (1. / (2 * m - 1));
}

// Rys nodes u_i = t_i^2 and weights: the large-x limit above xmax[N-1]
// (Gauss-Hermite); below it, for one to three roots the Gauss rule of the Boys
// moments (rows: load_moment_rows), else the Chebyshev tables.
template <int N>
__device__ __forceinline__ void rys_roots(const JKRysTable &tab, const lds_double *rows,
                                          double x, double *r, double *w)
{
    if (x >= tab.xmax[N-1]) {
        const double ix = rcp64(x), sx = rsqrt64(x);
        if constexpr (N <= 3) {
            constexpr double LR[6] = {0.5, 0.27525512860841095, 2.724744871391589,
                                      0.19016350919348812, 1.7844927485432516, 5.52534374226326};
            constexpr double LW[6] = {0.886226925452758, 0.8049140900055128, 0.08131283544724517,
                                      0.7246295952243925, 0.15706732032285664,
                                      0.004530009905508846};
#pragma unroll
            for (int i = 0; i < N; ++i) {
                r[i] = LR[N * (N - 1) / 2 + i] * ix;
                w[i] = LW[N * (N - 1) / 2 + i] * sx;
            }
        } else {
            const double *lr = tab.coef + tab.large_r + N * (N - 1) / 2;
            const double *lw = tab.coef + tab.large_w + N * (N - 1) / 2;
#pragma unroll
            for (int i = 0; i < N; ++i) { r[i] = lr[i] * ix; w[i] = lw[i] * sx; }
        }
        return;
    }
    if constexpr (N == 1) {
        double f[2];
        boys_moments<1>(rows, x, f);
        w[0] = f[0];
        r[0] = div64(f[1], f[0]);
        return;
    } else if constexpr (N == 2) {
        // monic p(u) = u^2 + c1 u + c0 orthogonal to 1 and u under the
        // moments: F2 + c1 F1 + c0 F0 = 0, F3 + c1 F2 + c0 F1 = 0
        // (c1 < 0: both nodes are positive)
        double f[4];
        boys_moments<2>(rows, x, f);
        const double idet = rcp64(f[1] * f[1] - f[0] * f[2]);
        const double c1 = (f[0] * f[3] - f[1] * f[2]) * idet;
        const double c0 = (f[2] * f[2] - f[1] * f[3]) * idet;
        const double disc = sqrt64(c1 * c1 - 4. * c0);
        const double u2 = .5 * (disc - c1), u1 = div64(c0, u2);
        const double w1 = div64(u2 * f[0] - f[1], u2 - u1);
        r[0] = u1; r[1] = u2;
        w[0] = w1; w[1] = f[0] - w1;
        return;
    } else if constexpr (N == 3) {
        // recurrence coefficients of the monic orthogonal polynomials from
        // the moments (Chebyshev's algorithm, Gautschi 2004, Alg. 2.1), the
        // nodes from Viete's trigonometric solution of the characteristic
        // cubic of the Jacobi matrix (in float: a starting point good to
        // 1e-5) refined by two Newton steps on the three-term recurrence
        // (1e-10, 1e-20), the weights by the Christoffel formula
        double mu[6];
        boys_moments<3>(rows, x, mu);
        const double r0 = rcp64(mu[0]);
        const double a0 = mu[1] * r0;
        const double n1 = mu[2] - a0 * mu[1], n2 = mu[3] - a0 * mu[2];
        const double n3 = mu[4] - a0 * mu[3], n4 = mu[5] - a0 * mu[4];
        const double rn1 = rcp64(n1);
        const double q1 = n2 * rn1, a1 = q1 - a0, b1 = n1 * r0;
        const double m2 = n3 - a1 * n2 - b1 * mu[2], m3 = n4 - a1 * n3 - b1 * mu[3];
        const double rm2 = rcp64(m2);
        const double a2 = m3 * rm2 - q1, b2 = m2 * rn1;
        const double c2 = -(a0 + a1 + a2);
        const double c1 = a0 * a1 + a0 * a2 + a1 * a2 - b1 - b2;
        const double c0 = b2 * a0 + b1 * a2 - a0 * a1 * a2;
        const double p = c1 - c2 * c2 * (1. / 3.);
        const double q = c2 * c2 * c2 * (2. / 27.) - c2 * c1 * (1. / 3.) + c0;
        const float rr = sqrtf((float)(-p) * (1.f / 3.f));
        const float phi = acosf(fminf(1.f, fmaxf(-1.f, -(float)q / (2.f * rr * rr * rr))));
        auto node = [&](float shift, double &rk, double &wk) {
            double v = (double)(2.f * rr * __cosf((phi + shift) * (1.f / 3.f))) - c2 * (1. / 3.);
            double p1, p2;
#pragma unroll
            for (int it = 0; it < 2; ++it) {
                p1 = v - a0;
                p2 = (v - a1) * p1 - b1;
                const double d2 = p1 + (v - a1);
                const double p3 = (v - a2) * p2 - b2 * p1, d3 = p2 + (v - a2) * d2 - b2;
                v -= p3 * __builtin_amdgcn_rcp(d3);
            }
            p1 = v - a0;
            p2 = (v - a1) * p1 - b1;
            // squared norms of the polynomials: mu_0, n1 = b0 b1, m2 = b0 b1 b2
            wk = rcp64(r0 + p1 * p1 * rn1 + p2 * p2 * rm2);
            rk = v;
        };
        // ascending: the node of phi + 2 pi is the smallest
        node(2.f * (float)M_PI, r[0], w[0]);
        node(-2.f * (float)M_PI, r[1], w[1]);
        node(0.f, r[2], w[2]);
        return;
    }
    const int D1 = tab.degree + 1;
    int k = (int)x;
    double u = 2. * (x - k) - 1.;
    double u2 = 2. * u;
    const double *c = tab.coef + tab.off[N-1] + (int64_t)k * (2 * N) * D1;
#pragma unroll
    for (int f = 0; f < 2 * N; ++f) {
        const double *cf = c + f * D1;
        double b1 = 0., b2 = 0.;
        for (int j = D1 - 1; j > 0; --j) {
            double t = fma(u2, b1, cf[j] - b2);
            b2 = b1; b1 = t;
        }
        double v = fma(u, b1, cf[0] - b2);
        if (f & 1) w[f >> 1] = v; else r[f >> 1] = v;
    }
}

// Root `i` and its weight only (one lane per root).
template <int N>
__device__ __forceinline__ void rys_root_one(const JKRysTable &tab, double x, int i,
                                             double &r, double &w)
{
    if (x >= tab.xmax[N-1]) {
        double ix = 1. / x;
        r = tab.coef[tab.large_r + N * (N - 1) / 2 + i] * ix;
        w = tab.coef[tab.large_w + N * (N - 1) / 2 + i] * sqrt(ix);
        return;
    }
    const int D1 = tab.degree + 1;
    int k = (int)x;
    double u = 2. * (x - k) - 1.;
    double u2 = 2. * u;
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

// runtime-N variant (setup kernels)
static __device__ void rys_roots_rt(const JKRysTable &tab, int N, double x, double *r, double *w)
{
    if (x >= tab.xmax[N-1]) {
        const double *lr = tab.coef + tab.large_r + N * (N - 1) / 2;
        const double *lw = tab.coef + tab.large_w + N * (N - 1) / 2;
        double ix = 1. / x, sx = sqrt(ix);
        for (int i = 0; i < N; ++i) { r[i] = lr[i] * ix; w[i] = lw[i] * sx; }
        return;
    }
    const int D1 = tab.degree + 1;
    int k = (int)x;
    double u = 2. * (x - k) - 1., u2 = 2. * u;
    const double *c = tab.coef + tab.off[N-1] + (int64_t)k * (2 * N) * D1;
    for (int f = 0; f < 2 * N; ++f) {
        const double *cf = c + f * D1;
        double b1 = 0., b2 = 0.;
        for (int j = D1 - 1; j > 0; --j) {
            double t = fma(u2, b1, cf[j] - b2);
            b2 = b1; b1 = t;
        }
        double v = fma(u, b1, cf[0] - b2);
        if (f & 1) w[f >> 1] = v; else r[f >> 1] = v;
    }
}

// 2D Rys integrals of one Cartesian direction for one root:
// g[((i*(LJ+1) + j)*(LK+1) + k)*(LL+1) + l], by VRR in i, TRR in k and HRR
// for j and l (the recursions of gpu4pyscf/lib/gvhf-rys/build_rys_gxyz.cuh:
// 18-123, evaluated in registers).
template <int LI, int LJ, int LK, int LL, typename T>
__device__ __forceinline__ void build_g(T *g, T g00, T c0, T cp, T b10, T b01, T b00,
                                        T rij, T rkl)
{
    constexpr int LIJ = LI + LJ, LKL = LK + LL;
    T G[LIJ+1][LKL+1];
    G[0][0] = g00;
    if (LIJ > 0) G[1][0] = c0 * g00;
#pragma unroll
    for (int a = 1; a < LIJ; ++a)
        G[a+1][0] = c0 * G[a][0] + ((T)a * b10) * G[a-1][0];
#pragma unroll
    for (int a = 0; a <= LIJ; ++a) {
        if (LKL > 0) {
            T v = cp * G[a][0];
            if (a > 0) v += ((T)a * b00) * G[a-1][0];
            G[a][1] = v;
        }
#pragma unroll
        for (int c = 1; c < LKL; ++c) {
            T v = cp * G[a][c] + ((T)c * b01) * G[a][c-1];
            if (a > 0) v += ((T)a * b00) * G[a-1][c];
            G[a][c+1] = v;
        }
    }
    // bra HRR: H[a][b][c] = H[a+1][b-1][c] - rij H[a][b-1][c]
    T H[LIJ+1][LJ+1][LKL+1];
#pragma unroll
    for (int c = 0; c <= LKL; ++c) {
#pragma unroll
        for (int a = 0; a <= LIJ; ++a) H[a][0][c] = G[a][c];
#pragma unroll
        for (int b = 0; b < LJ; ++b)
#pragma unroll
            for (int a = 0; a < LIJ - b; ++a)
                H[a][b+1][c] = H[a+1][b][c] - rij * H[a][b][c];
    }
    // ket HRR
#pragma unroll
    for (int a = 0; a <= LI; ++a)
#pragma unroll
    for (int b = 0; b <= LJ; ++b) {
        T W[LKL+1][LL+1];
#pragma unroll
        for (int c = 0; c <= LKL; ++c) W[c][0] = H[a][b][c];
#pragma unroll
        for (int e = 0; e < LL; ++e)
#pragma unroll
            for (int c = 0; c < LKL - e; ++c)
                W[c][e+1] = W[c+1][e] - rkl * W[c][e];
#pragma unroll
        for (int c = 0; c <= LK; ++c)
#pragma unroll
            for (int e = 0; e <= LL; ++e)
                g[((a*(LJ+1) + b)*(LK+1) + c)*(LL+1) + e] = W[c][e];
    }
}

// ---------------------------------------------------------------- shared
struct ShellPair {
    int ish, jsh, i0, j0;
    double ri[3], rij[3];      // Ri, Rj - Ri
    int pexpi, pexpj, pci, pcj;
};

__device__ __forceinline__ void load_shell_pair(ShellPair &s, uint32_t bas_ij, int nbas,
                                                const int32_t *bas, const double *env,
                                                const int32_t *ao_loc)
{
    s.ish = bas_ij / nbas;
    s.jsh = bas_ij - s.ish * nbas;
    const int32_t *bi = bas + s.ish * 8, *bj = bas + s.jsh * 8;
    const double *ri = env + bi[7], *rj = env + bj[7];
#pragma unroll
    for (int d = 0; d < 3; ++d) { s.ri[d] = ri[d]; s.rij[d] = rj[d] - ri[d]; }
    s.pexpi = bi[5]; s.pexpj = bj[5]; s.pci = bi[6]; s.pcj = bj[6];
    s.i0 = ao_loc[s.ish]; s.j0 = ao_loc[s.jsh];
}

// survival predicate, float32 in the reference's order: the bound test and
// pair order of create_tasks.cu:150-152, then the density blocks of the
// launch's screen (JKBuildArgs.screen): all six (:155-163), the Coulomb
// blocks D_ij, D_kl of a J-only build (:222-225) or the exchange blocks
// D_ik, D_jk, D_il, D_jl of a K-only build (:86-93)
// swapped (a launch with bra and ket exchanged, JKBuildArgs.swap_ijkl): the
// test in the task's own order and float32 rounding, with q_ij and cutoff
// the launch's bra bound and log(direct_scf_tol)
__device__ __forceinline__ bool survives(float q_kl, float kl_cutoff, float dm_penalty,
                                         uint32_t bas_ij, uint32_t bas_kl, int ish, int jsh,
                                         int nbas, const float *dm_cond, int screen,
                                         bool swapped = false, float q_ij = 0.f,
                                         float cutoff = 0.f)
{
    if (swapped) {
        kl_cutoff = cutoff - q_kl;
        q_kl = q_ij;
    }
    if (!(q_kl + dm_penalty >= kl_cutoff && (swapped ? bas_kl >= bas_ij : bas_ij >= bas_kl)))
        return false;
    int ksh = bas_kl / nbas;
    int lsh = bas_kl - ksh * nbas;
    float d_cutoff = kl_cutoff - q_kl;
    if (screen != JK_SCREEN_K &&
        (dm_cond[bas_ij] > d_cutoff || dm_cond[bas_kl] > d_cutoff))
        return true;
    // the exchange blocks D_ik, D_jk, D_il, D_jl of the task's shells
    const int ti = swapped ? ksh : ish, tj = swapped ? lsh : jsh;
    const int tk = swapped ? ish : ksh, tl = swapped ? jsh : lsh;
    return screen != JK_SCREEN_J &&
           (dm_cond[ti*nbas+tk] > d_cutoff ||
            dm_cond[tj*nbas+tk] > d_cutoff ||
            dm_cond[ti*nbas+tl] > d_cutoff ||
            dm_cond[tj*nbas+tl] > d_cutoff);
}

// SplitMix64 finaliser (Steele, Lea and Flood, OOPSLA 2014; constants of
// Vigna's splitmix64.c): the per-quartet term of the survivor set checksum
__device__ __forceinline__ unsigned long long quartet_mix(uint32_t bas_ij, uint32_t bas_kl);

// the checksum term of a quartet in the task's own order (bra and ket of a
// launch with swap_ijkl exchanged back)
__device__ __forceinline__ unsigned long long task_mix(const JKBuildArgs &a, uint32_t bas_ij,
                                                       uint32_t bas_kl)
{
    return a.swap_ijkl ? quartet_mix(bas_kl, bas_ij) : quartet_mix(bas_ij, bas_kl);
}

__device__ __forceinline__ unsigned long long quartet_mix(uint32_t bas_ij, uint32_t bas_kl)
{
    unsigned long long z = ((unsigned long long)bas_ij << 32) | bas_kl;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

// Same predicate, also returning the largest dm_cond value of the screen's
// blocks (any(v > d_cutoff) == max(v) > d_cutoff).
__device__ __forceinline__ bool survives_dmax(float q_kl, float kl_cutoff, float dm_penalty,
                                              uint32_t bas_ij, uint32_t bas_kl, int ish, int jsh,
                                              int nbas, const float *dm_cond, int screen,
                                              float &dmax, bool swapped = false,
                                              float q_ij = 0.f, float cutoff = 0.f)
{
    dmax = -1e30f;
    if (swapped) {
        kl_cutoff = cutoff - q_kl;
        q_kl = q_ij;
    }
    if (!(q_kl + dm_penalty >= kl_cutoff && (swapped ? bas_kl >= bas_ij : bas_ij >= bas_kl)))
        return false;
    int ksh = bas_kl / nbas;
    int lsh = bas_kl - ksh * nbas;
    float d_cutoff = kl_cutoff - q_kl;
    if (screen != JK_SCREEN_K)
        dmax = fmaxf(dm_cond[bas_ij], dm_cond[bas_kl]);
    // the exchange blocks D_ik, D_jk, D_il, D_jl of the task's shells
    const int ti = swapped ? ksh : ish, tj = swapped ? lsh : jsh;
    const int tk = swapped ? ish : ksh, tl = swapped ? jsh : lsh;
    if (screen != JK_SCREEN_J)
        dmax = fmaxf(dmax, fmaxf(fmaxf(dm_cond[ti*nbas+tk], dm_cond[tj*nbas+tk]),
                                 fmaxf(dm_cond[ti*nbas+tl], dm_cond[tj*nbas+tl])));
    return dmax > d_cutoff;
}

// Same predicate with the shells of kl and dm_cond[bas_ij] at hand.
__device__ __forceinline__ bool survives_sh(float q_kl, float kl_cutoff, float dm_penalty,
                                            uint32_t bas_ij, uint32_t bas_kl, int ish, int jsh,
                                            int ksh, int lsh, int nbas, const float *dm_cond,
                                            float dc_ij, int screen, bool swapped, float q_ij,
                                            float cutoff)
{
    if (swapped) {
        kl_cutoff = cutoff - q_kl;
        q_kl = q_ij;
    }
    if (!(q_kl + dm_penalty >= kl_cutoff && (swapped ? bas_kl >= bas_ij : bas_ij >= bas_kl)))
        return false;
    const float d_cutoff = kl_cutoff - q_kl;
    float dmax = -1e30f;
    if (screen != JK_SCREEN_K) dmax = fmaxf(dc_ij, dm_cond[bas_kl]);
    // the exchange blocks D_ik, D_jk, D_il, D_jl of the task's shells
    if (screen != JK_SCREEN_J) {
        const int s1 = swapped ? nbas : 1, sk = swapped ? 1 : nbas;
        const float *di = dm_cond + ish * sk, *dj = dm_cond + jsh * sk;
        dmax = fmaxf(dmax, fmaxf(fmaxf(di[ksh * s1], dj[ksh * s1]),
                                 fmaxf(di[lsh * s1], dj[lsh * s1])));
    }
    return dmax > d_cutoff;
}

// Work item of a launch: pair_ij index and the kl range of its chunk.
// One work item: ij pair pij against kl pairs [kl0, kl1), whose k and l AOs
// lie in [k_ao0, k_ao0 + k_nao) and [l_ao0, l_ao0 + l_nao) (the K-row
// columns of the item).
struct WorkItem { int pij, kl0, kl1, k_ao0, k_nao, l_ao0, l_nao; };

// use_lds bits of the per-lane and team kernels
#define KR_MODE_MASK    3       // 0 none, 1 K_il/K_jl rows, 2 all four K row blocks
#define KR_DROWS        4       // density rows staged too
#define KR_WIN          8       // work items = ij pairs x kl column windows

// A batched launch runs up to JK_BATCH tasks of one angular class: workgroup b
// belongs to the last task t with block0[t] <= b.  The class kernels of a
// small molecule are latency bound (one wavefront of quartets, a serial loop
// over the primitives), so what a build costs is the number of launches in a
// row: def2-SVP has 266 tasks but 21 angular classes, def2-TZVP 750 and 55.
// Building them class by class took one water molecule (def2-SVP) from 3.65 to
// 1.23 ms, 8 from 8.46 to 2.90 ms and 48 (def2-TZVP) from 1048 to 1020 ms.
// JK_BATCH descriptors and the shared arguments fill the 4 KB of kernel
// arguments, which reach the kernel through scalar loads; no descriptor is
// copied to device memory.
#define JK_BATCH 31
struct TaskDesc {
    const uint32_t *pairs_ij, *pairs_kl;
    const float *q_ij, *q_kl;
    const double *pdata_ij, *pdata_kl;
    const int32_t *win;             // kl column windows (KR_WIN)
    int npairs_ij, npairs_kl;
    uint32_t prims_ij, prims_kl;    // iprim | jprim << 16, kprim | lprim << 16
    int k_ao0, k_nao, l_ao0, l_nao;
    int kl_chunk;                   // candidates per work item (not KR_WIN)
    int use_lds;                    // KR_* bits
    int counter;                    // element of the per-task counters
    // li, lj, lk, ll, 4 bits each, swap_ijkl << 16, first density << 17
    uint32_t ls_swap;
};
struct TaskBatch {
    int n, pad;
    int block0[JK_BATCH + 1];       // first workgroup of each task, INT_MAX past n
    TaskDesc t[JK_BATCH];
};
static_assert(sizeof(JKBuildArgs) + sizeof(TaskBatch) + 64 <= 4096, "kernel arguments above 4 KB");

// A descriptor's pointer as one to global memory: the compiler takes that for
// granted for pointers among the kernel arguments, but not for those of a
// descriptor at a runtime index, whose accesses would become flat ones (no
// scalar base, 12 more registers and the LDS counter: (dp|ss) 18.4 -> 26.6 ms,
// (fp|dp) 34 -> 52 ms of the 48-water def2-TZVP build).
template <typename T>
__device__ __forceinline__ T *as_global(T *p)
{
    return (T *)(__attribute__((address_space(1))) T *)p;
}

// The task of this workgroup: its fields into the launch's arguments;
// returns the workgroup's index within the task.
__device__ __forceinline__ int select_task(JKBuildArgs &a, const TaskBatch &b, int &kl_chunk,
                                           int &use_lds, int &dm0)
{
    const int blk = blockIdx.x;
    int t = 0;
#pragma unroll
    for (int n = 1; n < JK_BATCH; ++n) t = blk >= b.block0[n] ? n : t;
    const TaskDesc &d = b.t[t];
    a.li = d.ls_swap & 15; a.lj = d.ls_swap >> 4 & 15;
    a.lk = d.ls_swap >> 8 & 15; a.ll = d.ls_swap >> 12 & 15;
    a.swap_ijkl = d.ls_swap >> 16 & 1;
    dm0 = d.ls_swap >> 17;
    a.pairs_ij = as_global(d.pairs_ij); a.pairs_kl = as_global(d.pairs_kl);
    a.q_ij = as_global(d.q_ij); a.q_kl = as_global(d.q_kl);
    a.pdata_ij = as_global(d.pdata_ij); a.pdata_kl = as_global(d.pdata_kl);
    a.kl_win[0].win = as_global(d.win);
    a.npairs_ij = d.npairs_ij; a.npairs_kl = d.npairs_kl;
    a.iprim = d.prims_ij & 0xffff; a.jprim = d.prims_ij >> 16;
    a.kprim = d.prims_kl & 0xffff; a.lprim = d.prims_kl >> 16;
    a.k_ao0 = d.k_ao0; a.k_nao = d.k_nao; a.l_ao0 = d.l_ao0; a.l_nao = d.l_nao;
    // (the launches of the first density count)
    a.n_quartets = a.n_quartets && dm0 == 0 ? a.n_quartets + d.counter : nullptr;
    a.n_quartets_fp32 = a.n_quartets_fp32 && dm0 == 0 ? a.n_quartets_fp32 + d.counter : nullptr;
    a.quartet_hash = a.quartet_hash && dm0 == 0 ? a.quartet_hash + d.counter : nullptr;
    kl_chunk = d.kl_chunk;
    use_lds = d.use_lds;
    return blk - b.block0[t];
}

__device__ __forceinline__ int select_task(JKBuildArgs &a, const TaskBatch &b, int &kl_chunk,
                                           int &use_lds)
{
    int dm0;
    return select_task(a, b, kl_chunk, use_lds, dm0);
}

__device__ __forceinline__ WorkItem work_item(int idx, int npairs_kl, int kl_chunk)
{
    int nchunks = (npairs_kl + kl_chunk - 1) / kl_chunk;
    WorkItem w;
    w.pij = idx / nchunks;
    int ch = idx - w.pij * nchunks;
    w.kl0 = ch * kl_chunk;
    w.kl1 = min(w.kl0 + kl_chunk, npairs_kl);
    w.k_ao0 = w.k_nao = w.l_ao0 = w.l_nao = 0;
    return w;
}

// work items over the kl column windows of kl_win[0] (window major, ij pair
// minor; the launcher puts the team kernels' set there); the K-row columns
// are the window's
__device__ __forceinline__ WorkItem work_item_win(const JKBuildArgs &a, int idx)
{
    WorkItem w;
    const int win = idx / a.npairs_ij;
    w.pij = idx - win * a.npairs_ij;
    const int32_t *d = a.kl_win[0].win + 6 * win;
    w.kl0 = d[0]; w.kl1 = d[1];
    w.k_ao0 = d[2]; w.k_nao = d[3]; w.l_ao0 = d[4]; w.l_nao = d[5];
    return w;
}

// work item idx of a per-lane or team task: kl chunks over the whole groups,
// or the kl column windows
__device__ __forceinline__ WorkItem work_item(const JKBuildArgs &a, int idx, int kl_chunk,
                                              int use_lds)
{
    if (use_lds & KR_WIN) return work_item_win(a, idx);
    WorkItem w = work_item(idx, a.npairs_kl, kl_chunk);
    w.k_ao0 = a.k_ao0; w.k_nao = a.k_nao; w.l_ao0 = a.l_ao0; w.l_nao = a.l_nao;
    return w;
}

// K rows of one work item accumulated in LDS (one density): rows i (NFI)
// then j (NFJ); columns: the work item's k AOs (when kcols) followed by its
// l AOs (the whole k and l groups, or one kl column window).  Flushed to K with one atomic per non-zero element.
// The same row layout also holds, after the K rows, a copy of the density
// rows i and j over the k and l group columns (dstaged), from which the
// per-lane digestion reads D_ik, D_il, D_jk and D_jl.
// p and d always point into the LDS array; `on` and `dstaged` say whether they
// are used.
struct KRows {
    lds_double *p;          // K rows
    const lds_double *d;    // density rows
    int width;          // doubles per row
    int loff;           // column of the first l AO
    int k_ao0, l_ao0;   // AOs of columns 0 and loff
    bool on;            // K_il / K_jl (and with kcols K_ik / K_jk) accumulated here
    bool kcols;         // K_ik / K_jk accumulated here too
    bool dstaged;       // density rows present
};

// use_lds: 0 none, 1 K_il/K_jl rows, 2 K_ik/K_jk and K_il/K_jl rows,
// 2|4 the same plus the density rows
__device__ __forceinline__ KRows make_krows(double *buf, int use_lds, int nrows,
                                            const WorkItem &w)
{
    KRows kr;
    kr.on = (use_lds & KR_MODE_MASK) != 0;
    kr.kcols = (use_lds & KR_MODE_MASK) == 2;
    kr.dstaged = kr.kcols && (use_lds & KR_DROWS);
    kr.loff = kr.kcols ? w.k_nao : 0;
    kr.width = kr.loff + w.l_nao;
    kr.k_ao0 = w.k_ao0;
    kr.l_ao0 = w.l_ao0;
    kr.p = (lds_double *)buf;
    kr.d = kr.p + nrows * kr.width;
    return kr;
}

// the same rows `off` doubles on (another density's)
__device__ __forceinline__ KRows krows_of(KRows kr, int off)
{
    kr.p += off;
    kr.d += off;
    return kr;
}

// copy the density rows (after krows_zero; a barrier must follow)
__device__ __forceinline__ void krows_load_d(const KRows &kr, int nfi, int nfj, int i0, int j0,
                                             int nao, const double *dm, int tid, int nthreads)
{
    if (!kr.dstaged) return;
    lds_double *d = kr.p + (nfi + nfj) * kr.width;
    const int n_all = (nfi + nfj) * kr.width;
    for (int n = tid; n < n_all; n += nthreads) {
        int r = n / kr.width, c = n - r * kr.width;
        int row = r < nfi ? i0 + r : j0 + r - nfi;
        int col = c < kr.loff ? kr.k_ao0 + c : kr.l_ao0 + c - kr.loff;
        d[n] = dm[(size_t)row * nao + col];
    }
}

// zero (before the block's first quartet; a barrier must follow)
__device__ __forceinline__ void krows_zero(const KRows &kr, int nrows, int tid, int nthreads)
{
    if (!kr.on) return;
    for (int n = tid; n < nrows * kr.width; n += nthreads) kr.p[n] = 0.;
}

// flush (after a barrier that ends the block's accumulation)
__device__ __forceinline__ void krows_flush(const KRows &kr, int nfi, int nfj, int i0, int j0,
                                            int nao, double *vk, int tid, int nthreads)
{
    if (!kr.on) return;
    const int n_all = (nfi + nfj) * kr.width;
    for (int n = tid; n < n_all; n += nthreads) {
        double v = kr.p[n];
        if (v != 0.) {
            int r = n / kr.width, c = n - r * kr.width;
            int row = r < nfi ? i0 + r : j0 + r - nfi;
            int col = c < kr.loff ? kr.k_ao0 + c : kr.l_ao0 + c - kr.loff;
            atomic_add(vk + (size_t)row * nao + col, v);
        }
    }
}

// ---------------------------------------------------------------- per-lane
// Primitive-pair record, see jk_pair_data(): (a, 1/a, Px, Py, Pz, K).
#define PREC 6

// Rys roots in FP32: Chebyshev series in float on the float copy of the
// table; the large-x asymptotic branch is evaluated in FP64.
template <int N>
__device__ __forceinline__ void rys_roots(const JKRysTable &tab, const lds_double *, float x,
                                          float *r, float *w)
{
    if (x >= (float)tab.xmax[N-1]) {
        double xd = x;
        const double *lr = tab.coef + tab.large_r + N * (N - 1) / 2;
        const double *lw = tab.coef + tab.large_w + N * (N - 1) / 2;
        double ix = 1. / xd;
        double sx = sqrt(ix);
#pragma unroll
        for (int i = 0; i < N; ++i) { r[i] = (float)(lr[i] * ix); w[i] = (float)(lw[i] * sx); }
        return;
    }
    const int D1 = tab.degree + 1;
    int k = (int)x;
    float u = 2.f * (x - k) - 1.f;
    float u2 = 2.f * u;
    const float *c = tab.coef32 + tab.off[N-1] + (int64_t)k * (2 * N) * D1;
#pragma unroll
    for (int f = 0; f < 2 * N; ++f) {
        const float *cf = c + f * D1;
        float b1 = 0.f, b2 = 0.f;
        for (int j = D1 - 1; j > 0; --j) {
            float t = fmaf(u2, b1, cf[j] - b2);
            b2 = b1; b1 = t;
        }
        float v = fmaf(u, b1, cf[0] - b2);
        if (f & 1) w[f >> 1] = v; else r[f >> 1] = v;
    }
}

// The primitives of the (uniform) ij pair: a, 1/a, P, K, P - R_i of record ip,
// from the pair records in HBM or from their copy in LDS (stage_pij).
#define PIJ_LDS 10      // doubles of one primitive's copy
struct PijGlobal {
    const double *rec, *ri;
    __device__ __forceinline__ void get(int ip, double &a, double &ra, double *P, double &K,
                                        double *PA) const
    {
        const double *p = rec + ip * PREC;
        a = p[0]; ra = p[1]; K = p[5];
#pragma unroll
        for (int d = 0; d < 3; ++d) { P[d] = p[2+d]; PA[d] = p[2+d] - ri[d]; }
    }
};

struct PijLds {
    const lds_double *rec;
    __device__ __forceinline__ void get(int ip, double &a, double &ra, double *P, double &K,
                                        double *PA) const
    {
        const lds_double2 *p = (const lds_double2 *)(rec + ip * PIJ_LDS);
        const double2v v0 = p[0], v1 = p[1], v2 = p[2], v3 = p[3], v4 = p[4];
        a = v0.x; ra = v0.y;
        P[0] = v1.x; P[1] = v1.y; P[2] = v2.x; K = v2.y;
        PA[0] = v3.x; PA[1] = v3.y; PA[2] = v4.x;
    }
};

// copies the records of the work item's ij pair (a barrier must follow)
__device__ __forceinline__ void stage_pij(lds_double *dst, const double *rec, int nij,
                                          const double *ri, int tid, int nthreads)
{
    for (int n = tid; n < nij; n += nthreads) {
        const double *p = rec + n * PREC;
        lds_double *o = dst + n * PIJ_LDS;
        o[0] = p[0]; o[1] = p[1]; o[2] = p[2]; o[3] = p[3]; o[4] = p[4]; o[5] = p[5];
        o[6] = p[2] - ri[0]; o[7] = p[3] - ri[1]; o[8] = p[4] - ri[2];
    }
}

// Operator of a launch (JKBuildArgs.omega, full): erf(omega r)/r for omega2 > 0,
// else 1/r; with full != 0 also full / r, as a second set of roots of every
// primitive quartet.  The two parts of a range-separated operator then share
// screening, primitives, densities and the additions into K (range-separated K
// of 16 waters def2-TZVP 131 -> 97 ms).  DUAL: the kernel may be given a second
// part; the per-lane kernels with J are not: a loop around one part kept the
// compiler from scheduling across it ((pp|ss) 150 -> 168 us, (ss|ss) 246 -> 275
// of 8 waters def2-SVP), and there two launches serve.
template <bool DUAL>
struct Oper {
    double omega2, full;
    __device__ __forceinline__ explicit Oper(const JKBuildArgs &a)
        : omega2(a.omega * a.omega), full(DUAL ? a.full : 0.) {}
    __device__ __forceinline__ int parts() const { return DUAL && full != 0. ? 2 : 1; }
};

// One quartet per lane in arithmetic type T (double or float): returns the
// rows I0 <= i < I1 of the Cartesian block (times the symmetry and
// normalisation prefactors) in gout[(((i-I0)*nfj+j)*nfk+k)*nfl+l].
// pij: the primitives of the (uniform) ij pair; pkl: records of this lane's kl
// pair.  `loaded` is called once, when the first kl record has arrived.
template <int LI, int LJ, int LK, int LL, typename T, int I0 = 0, int I1 = ncart(LI),
          bool DUAL = false, typename Pij, typename F>
__device__ __forceinline__ void eri_lane(T *gout, const Pij &pij, int nij,
                                         const double *pkl, int nkl, const double *rij,
                                         const double *rk, const double *rkl,
                                         const JKRysTable &rys, const lds_double *rows,
                                         double fac_sym, const Oper<DUAL> &op, F &&loaded)
{
    constexpr int NFJ = ncart(LJ), NFK = ncart(LK), NFL = ncart(LL);
    constexpr int NF = (I1 - I0) * NFJ * NFK * NFL;
    constexpr int N = (LI + LJ + LK + LL) / 2 + 1;
    constexpr int GS = (LI+1)*(LJ+1)*(LK+1)*(LL+1);
    constexpr CartPow<LI> ci{};
    constexpr CartPow<LJ> cj{};
    constexpr CartPow<LK> ck{};
    constexpr CartPow<LL> cl{};
    const T rij_t[3] = {(T)rij[0], (T)rij[1], (T)rij[2]};
    const T rkl_t[3] = {(T)rkl[0], (T)rkl[1], (T)rkl[2]};
#pragma unroll
    for (int n = 0; n < NF; ++n) gout[n] = 0;
    double q[PREC];
#pragma unroll
    for (int n = 0; n < PREC; ++n) q[n] = pkl[n];
    loaded();
    for (int kp = 0; kp < nkl; ++kp) {
        if (kp > 0) {
#pragma unroll
            for (int n = 0; n < PREC; ++n) q[n] = pkl[kp * PREC + n];
        }
        const T akl = (T)q[0], rakl = (T)q[1];
        const T Kkl = (T)(q[5] * fac_sym);
        T QC[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) QC[d] = (T)(q[2+d] - rk[d]);
        for (int ip = 0; ip < nij; ++ip) {
            double a_d, ra_d, P_d[3], K_d, PA_d[3];
            pij.get(ip, a_d, ra_d, P_d, K_d, PA_d);
            const T aij = (T)a_d, raij = (T)ra_d;
            T PA[3], PQ[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                PA[d] = (T)PA_d[d];
                PQ[d] = (T)(P_d[d] - q[2+d]);
            }
            T rr = PQ[0]*PQ[0] + PQ[1]*PQ[1] + PQ[2]*PQ[2];
            T r_aa = rcp64(aij + akl);
            T theta = aij * akl * r_aa;
            T fac = (T)K_d * Kkl * rsqrt64(aij + akl);
            auto add_part = [&](double omega2, T fac) {
                T rt[N], wt[N];
                // long-range attenuation erf(omega r)/r: the rule at x a with the
                // roots scaled by a and the weights by sqrt(a)
                T aw = (T)1;
                if (omega2 > 0.) aw = (T)omega2 / ((T)omega2 + theta);
                if constexpr (sizeof(T) == sizeof(float) && N <= 3) {
                    // the rule of the Boys moments in FP64 is cheaper than the float
                    // Chebyshev series for up to three roots
                    double rd[N], wd[N];
                    rys_roots<N>(rys, rows, (double)(theta * rr * aw), rd, wd);
#pragma unroll
                    for (int i = 0; i < N; ++i) { rt[i] = (T)rd[i]; wt[i] = (T)wd[i]; }
                } else {
                    rys_roots<N>(rys, rows, theta * rr * aw, rt, wt);
                }
                if (omega2 > 0.) {
                    const T sa = sqrt(aw);
#pragma unroll
                    for (int i = 0; i < N; ++i) { rt[i] *= aw; wt[i] *= sa; }
                }
#pragma unroll
                for (int ir = 0; ir < N; ++ir) {
                    T rt_aa = rt[ir] * r_aa;
                    T rt_aij = rt_aa * akl, rt_akl = rt_aa * aij;
                    T b10 = (T).5 * raij * ((T)1 - rt_aij);
                    T b01 = (T).5 * rakl * ((T)1 - rt_akl);
                    T b00 = (T).5 * rt_aa;
                    T gx[GS], gy[GS], gz[GS];
                    build_g<LI, LJ, LK, LL>(gx, (T)1, PA[0] - rt_aij * PQ[0], QC[0] + rt_akl * PQ[0],
                                            b10, b01, b00, rij_t[0], rkl_t[0]);
                    build_g<LI, LJ, LK, LL>(gy, (T)1, PA[1] - rt_aij * PQ[1], QC[1] + rt_akl * PQ[1],
                                            b10, b01, b00, rij_t[1], rkl_t[1]);
                    build_g<LI, LJ, LK, LL>(gz, wt[ir] * fac, PA[2] - rt_aij * PQ[2],
                                            QC[2] + rt_akl * PQ[2], b10, b01, b00, rij_t[2], rkl_t[2]);
#pragma unroll
                    for (int i = I0; i < I1; ++i)
#pragma unroll
                    for (int j = 0; j < NFJ; ++j)
#pragma unroll
                    for (int k = 0; k < NFK; ++k)
#pragma unroll
                    for (int l = 0; l < NFL; ++l) {
                        constexpr int SJ = LL+1, SK = (LK+1)*(LL+1), SI = (LJ+1)*(LK+1)*(LL+1);
                        int ix = ci.x[i]*SI + cj.x[j]*SK + ck.x[k]*SJ + cl.x[l];
                        int iy = ci.y[i]*SI + cj.y[j]*SK + ck.y[k]*SJ + cl.y[l];
                        int iz = ci.z[i]*SI + cj.z[j]*SK + ck.z[k]*SJ + cl.z[l];
                        int n = (((i - I0)*NFJ + j)*NFK + k)*NFL + l;
                        gout[n] = fma(gx[ix] * gy[iy], gz[iz], gout[n]);
                    }
                }
            };
            if constexpr (DUAL) {
#pragma unroll 1
                for (int part = op.parts() - 1; part >= 0; --part)
                    add_part(part ? 0. : op.omega2, part ? fac * (T)op.full : fac);
            } else {
                add_part(op.omega2, fac);
            }
        }
    }
}

// Rows of the Cartesian block a per-lane quartet holds in registers at a
// time: all NFI when the block and three 2D tables fit in LANE_MAX doubles,
// else chunks of CH rows i (each chunk re-evaluates the roots and 2D tables).
// Doubles of one chunk (its rows of the block plus three 2D tables) per
// class: LANE_CHUNK_MAX, or more where three larger chunks measured faster
// than five smaller ones (64-water build, ms on one stream: (fp|pp) 77.2 ->
// 60.7, (ff|ps) -> 50.5 against 55.5 on teams, (fp|fs) on 32 waters 10.6
// against 11.6 on teams).
template <int LI, int LJ, int LK, int LL> struct LaneChunkBudget {
    static constexpr int D = LANE_CHUNK_MAX;
};
#define LANE_CHUNK_BUDGET(a, b, c, d, n) \
    template <> struct LaneChunkBudget<a, b, c, d> { static constexpr int D = n; };
LANE_CHUNK_BUDGET(3, 1, 1, 1, 220) LANE_CHUNK_BUDGET(3, 3, 1, 0, 220)
LANE_CHUNK_BUDGET(3, 1, 3, 0, 220)
#undef LANE_CHUNK_BUDGET

template <int LI, int LJ, int LK, int LL>
struct LaneChunk {
    static constexpr int NFI = ncart(LI);
    static constexpr int ROW = ncart(LJ) * ncart(LK) * ncart(LL);
    static constexpr int GS3 = 3 * (LI+1)*(LJ+1)*(LK+1)*(LL+1);
    static constexpr int FIT = (LaneChunkBudget<LI, LJ, LK, LL>::D - GS3) / ROW;
    static constexpr int CH = NFI * ROW + GS3 <= LANE_MAX ? NFI : (FIT > 0 ? FIT : 1);
    static constexpr int NCH = (NFI + CH - 1) / CH;
};

// Classes above LANE_MAX that run per lane in chunks: those measured faster
// than on teams (64-water def2-TZVP build, ms on one stream, team ->
// chunked lanes: (fp|ds) 91.6 -> 54.4, (fd|ps) 85.0 -> 39.1, (dp|pp) 69.9 ->
// 52.5, (dd|ds) 37.6 -> 12.7, (fp|pp) 70.1 -> 60.7 and (ff|ps) 55.5 -> 50.5
// with the larger chunks of LaneChunkBudget; 32-water alike).  Slower per
// lane and left on teams: (fs|dp) 65.9 -> 73.6, (fs|fp) 40.3 -> 68.2,
// (ds|dd) 8.4 -> 34.9.
template <int LI, int LJ, int LK, int LL> struct LaneChunked { static constexpr bool ON = false; };
#define LANE_CHUNKED(a, b, c, d) \
    template <> struct LaneChunked<a, b, c, d> { static constexpr bool ON = true; };
LANE_CHUNKED(3, 1, 2, 0) LANE_CHUNKED(3, 2, 1, 0) LANE_CHUNKED(2, 1, 1, 1) LANE_CHUNKED(2, 2, 2, 0)
LANE_CHUNKED(3, 1, 1, 1) LANE_CHUNKED(3, 3, 1, 0) LANE_CHUNKED(3, 1, 3, 0)
#undef LANE_CHUNKED

// f(std::integral_constant<int, c>()) for c = 0 .. NC-1, unrolled at compile time
template <int C, int NC>
struct LaneChunkLoop {
    template <typename F>
    __device__ __forceinline__ static void run(F &f)
    {
        f(std::integral_constant<int, C>());
        LaneChunkLoop<C + 1, NC>::run(f);
    }
};
template <int NC>
struct LaneChunkLoop<NC, NC> {
    template <typename F>
    __device__ __forceinline__ static void run(F &) {}
};
template <int NC, typename F>
__device__ __forceinline__ void lane_chunks(F &&f)
{
    LaneChunkLoop<0, NC>::run(f);
}

// Evaluates and digests one batch of up to 64 queued quartets (one per lane)
// in arithmetic type T; digestion and accumulation are FP64.
template <int LI, int LJ, int LK, int LL, typename T>
__device__ __forceinline__ void lane_batch(const JKBuildArgs &a, const ShellPair &sp,
                                           uint32_t bas_ij, int pij, const uint32_t *queue,
                                           int nb, int lane, uint64_t lt_mask, const KRows &kr,
                                           const lds_double *rows)
{
    constexpr int NFI = ncart(LI), NFJ = ncart(LJ), NFK = ncart(LK), NFL = ncart(LL);
    constexpr int CH = LaneChunk<LI, LJ, LK, LL>::CH;
    const int nbas = a.nbas, nao = a.nao;
    const size_t nao2 = (size_t)nao * nao;
    const bool active = lane < nb;
    const int pkl = queue[active ? lane : 0];
    const uint32_t bas_kl = a.pairs_kl[pkl];
    const int ksh = bas_kl / nbas, lsh = bas_kl - (bas_kl / nbas) * nbas;
    double fac_sym = a.scale;
    if (sp.ish == sp.jsh) fac_sym *= .5;
    if (ksh == lsh) fac_sym *= .5;
    if (bas_ij == bas_kl) fac_sym *= .5;
    if (!active) fac_sym = 0.;
    const double *rk = a.env + a.bas[ksh * 8 + 7], *rl = a.env + a.bas[lsh * 8 + 7];
    const double rk3[3] = {rk[0], rk[1], rk[2]};
    const double rkl[3] = {rl[0] - rk[0], rl[1] - rk[1], rl[2] - rk[2]};
    const int nij = a.iprim * a.jprim, nkl = a.kprim * a.lprim;
    const int k0 = a.ao_loc[ksh], l0 = a.ao_loc[lsh];
    const int i0 = sp.i0, j0 = sp.j0;
    // runs of equal k shell are contiguous in the queue (tile order):
    // segment = run id, from the run heads
    const int key = active ? ksh : -1;
    const int key_prev = __shfl_up(key, 1, WAVE);
    const bool head = lane == 0 || key_prev != key;
    const uint64_t heads = __ballot(head);
    const int run = __popcll(heads & (lt_mask | (1ull << lane)));
    const int run_next = __shfl_down(run, 1, WAVE);
    const bool tail = active && (lane == nb - 1 || run_next != run);
    const SegMask runs = seg_mask(run, lane);
    // columns of this quartet's k and l AOs in the LDS density rows
    const int dk = k0 - kr.k_ao0, dl = kr.loff + l0 - kr.l_ao0;
    // rows i of the block in chunks of CH (one chunk unless the block and
    // its 2D tables would not fit the registers): evaluate, then digest
    lane_chunks<(NFI + CH - 1) / CH>([&](auto cc) {
        constexpr int I0 = decltype(cc)::value * CH;
        constexpr int I1 = I0 + CH < NFI ? I0 + CH : NFI;
        constexpr int NI = I1 - I0;
        T gout[NI * NFJ * NFK * NFL];
        eri_lane<LI, LJ, LK, LL, T, I0, I1>(
            gout, PijGlobal{a.pdata_ij + (size_t)pij * nij * PREC, sp.ri}, nij,
            a.pdata_kl + (size_t)pkl * nkl * PREC, nkl, sp.rij, rk3, rkl, a.rys, rows, fac_sym,
            Oper<false>(a), [] {});
        for (int id = 0; id < a.n_dm; ++id) {
            const double *D = a.dm + id * nao2;
            if (a.vk) {
                double *K = a.vk + id * nao2;
                // K_ik += (ij|kl) D_jl ; K_il += (ij|kl) D_jk
#pragma unroll
                for (int i = I0; i < I1; ++i) {
                    double kil[NFL], kik[NFK];
#pragma unroll
                    for (int l = 0; l < NFL; ++l) kil[l] = 0.;
#pragma unroll
                    for (int k = 0; k < NFK; ++k) kik[k] = 0.;
                    if (active && kr.dstaged) {
#pragma unroll
                        for (int j = 0; j < NFJ; ++j)
#pragma unroll
                        for (int k = 0; k < NFK; ++k)
#pragma unroll
                        for (int l = 0; l < NFL; ++l) {
                            double g = gout[(((i - I0)*NFJ + j)*NFK + k)*NFL + l];
                            kil[l] = fma(g, kr.d[(NFI + j) * kr.width + dk + k], kil[l]);
                            kik[k] = fma(g, kr.d[(NFI + j) * kr.width + dl + l], kik[k]);
                        }
                    } else if (active) {
#pragma unroll
                        for (int j = 0; j < NFJ; ++j)
#pragma unroll
                        for (int k = 0; k < NFK; ++k)
#pragma unroll
                        for (int l = 0; l < NFL; ++l) {
                            double g = gout[(((i - I0)*NFJ + j)*NFK + k)*NFL + l];
                            kil[l] = fma(g, D[(j0+j)*nao + k0+k], kil[l]);
                            kik[k] = fma(g, D[(j0+j)*nao + l0+l], kik[k]);
                        }
                    }
                    if (kr.kcols && LANE_KIK_SEGSUM) {
#pragma unroll
                        for (int k = 0; k < NFK; ++k) {
                            double v = seg_sum(kik[k], runs);
                            if (tail) lds_add(kr.p + i * kr.width + k0 + k - kr.k_ao0, v);
                        }
                    } else if (kr.kcols) {
                        if (active) {
#pragma unroll
                            for (int k = 0; k < NFK; ++k)
                                lds_add(kr.p + i * kr.width + k0 + k - kr.k_ao0, kik[k]);
                        }
                    } else {
#pragma unroll
                        for (int k = 0; k < NFK; ++k) {
                            double v = seg_sum(kik[k], runs);
                            if (tail) atomic_add(K + (i0+i)*nao + k0+k, v);
                        }
                    }
                    if (active) {
#pragma unroll
                        for (int l = 0; l < NFL; ++l) {
                            if (kr.on) lds_add(kr.p + i * kr.width + kr.loff + l0 + l - kr.l_ao0, kil[l]);
                            else atomic_add(K + (i0+i)*nao + l0+l, kil[l]);
                        }
                    }
                }
                // K_jk += (ij|kl) D_il ; K_jl += (ij|kl) D_ik
#pragma unroll
                for (int j = 0; j < NFJ; ++j) {
                    double kjl[NFL], kjk[NFK];
#pragma unroll
                    for (int l = 0; l < NFL; ++l) kjl[l] = 0.;
#pragma unroll
                    for (int k = 0; k < NFK; ++k) kjk[k] = 0.;
                    if (active && kr.dstaged) {
#pragma unroll
                        for (int i = I0; i < I1; ++i)
#pragma unroll
                        for (int k = 0; k < NFK; ++k)
#pragma unroll
                        for (int l = 0; l < NFL; ++l) {
                            double g = gout[(((i - I0)*NFJ + j)*NFK + k)*NFL + l];
                            kjl[l] = fma(g, kr.d[i * kr.width + dk + k], kjl[l]);
                            kjk[k] = fma(g, kr.d[i * kr.width + dl + l], kjk[k]);
                        }
                    } else if (active) {
#pragma unroll
                        for (int i = I0; i < I1; ++i)
#pragma unroll
                        for (int k = 0; k < NFK; ++k)
#pragma unroll
                        for (int l = 0; l < NFL; ++l) {
                            double g = gout[(((i - I0)*NFJ + j)*NFK + k)*NFL + l];
                            kjl[l] = fma(g, D[(i0+i)*nao + k0+k], kjl[l]);
                            kjk[k] = fma(g, D[(i0+i)*nao + l0+l], kjk[k]);
                        }
                    }
                    if (kr.kcols && LANE_KIK_SEGSUM) {
#pragma unroll
                        for (int k = 0; k < NFK; ++k) {
                            double v = seg_sum(kjk[k], runs);
                            if (tail) lds_add(kr.p + (NFI + j) * kr.width + k0 + k - kr.k_ao0, v);
                        }
                    } else if (kr.kcols) {
                        if (active) {
#pragma unroll
                            for (int k = 0; k < NFK; ++k)
                                lds_add(kr.p + (NFI + j) * kr.width + k0 + k - kr.k_ao0, kjk[k]);
                        }
                    } else {
#pragma unroll
                        for (int k = 0; k < NFK; ++k) {
                            double v = seg_sum(kjk[k], runs);
                            if (tail) atomic_add(K + (j0+j)*nao + k0+k, v);
                        }
                    }
                    if (active) {
#pragma unroll
                        for (int l = 0; l < NFL; ++l) {
                            if (kr.on) lds_add(kr.p + (NFI + j) * kr.width + kr.loff + l0 + l - kr.l_ao0, kjl[l]);
                            else atomic_add(K + (j0+j)*nao + l0+l, kjl[l]);
                        }
                    }
                }
            }
            if (a.vj) {
                double *J = a.vj + id * nao2;
                // the D_kl loads of J_ij come before the J_kl atomics: on this GPU
                // stores and atomics share the load counter, so a load issued
                // after an atomic waits for it to complete.
                // J_ij partial sums of this lane (D_kl): reduced over the wave below
                double vij[NI*NFJ];
#pragma unroll
                for (int i = I0; i < I1; ++i)
#pragma unroll
                for (int j = 0; j < NFJ; ++j) {
                    double s = 0.;
                    if (active) {
#pragma unroll
                        for (int k = 0; k < NFK; ++k)
#pragma unroll
                        for (int l = 0; l < NFL; ++l)
                            s = fma((double)gout[(((i - I0)*NFJ + j)*NFK + k)*NFL + l],
                                    D[(k0+k)*nao + l0+l], s);
                    }
                    vij[(i - I0)*NFJ + j] = s;
                }
                // J_kl += (ij|kl) D_ij   (per lane)
                if (active) {
#pragma unroll
                    for (int k = 0; k < NFK; ++k)
#pragma unroll
                    for (int l = 0; l < NFL; ++l) {
                        double s = 0.;
#pragma unroll
                        for (int i = I0; i < I1; ++i)
#pragma unroll
                        for (int j = 0; j < NFJ; ++j)
                            s = fma((double)gout[(((i - I0)*NFJ + j)*NFK + k)*NFL + l],
                                    D[(i0+i)*nao + j0+j], s);
                        atomic_add(J + (k0+k)*nao + l0+l, s);
                    }
                }
                // J_ij += (ij|kl) D_kl   (common ij: reduce over the wave)
                wave_reduce_scatter<NI*NFJ>(vij, lane, [&](int n, double x) {
                    atomic_add(J + (i0 + I0 + n / NFJ)*nao + j0 + n % NFJ, x);
                });
            }
        }
    });
}

// Per-lane kernel.  NW wavefronts share one work item (and its LDS K
// rows); each wavefront scans every NW-th batch of 64 kl candidates
// and keeps two queues: quartets whose bound q_ij + q_kl + max(dm_cond)
// reaches fp32_cut run in FP64, the others in FP32.  PM (precision mode):
// 0 both queues, 1 the FP64 queue only, 2 the FP32 queue only (a launch
// with PM 1 and one with PM 2 together evaluate what one with PM 0 does;
// each is compiled without the other's arithmetic).  FP64 builds launch PM 1
// (64-water build 2110 -> 2092 ms against PM 0); mixed builds PM 0, since
// the pair PM 1 + PM 2 scans and flushes every work item twice (2115 ->
// 2253 ms; the FP32-only kernels mostly keep the occupancy of PM 0).
// Wavefronts per workgroup of the per-lane kernels.  The K and density rows of a
// work item are LDS that its wavefronts share: four of them where the registers
// leave room for more wavefronts than the rows of two-wave workgroups do.
// 48 waters (def2-TZVP), one stream, ms, two waves -> four: (ps|ss) 58.5 -> 50.7,
// (fs|ps) 37.3 -> 31.4, (ff|ps) 24.9 -> 19.5, (ds|ss) 24.5 -> 19.1, (fs|ss)
// 20.9 -> 16.1, (pp|ss) 19.9 -> 14.7, (fp|ss) 19.4 -> 17.2, (ff|ss) 16.4 -> 12.1,
// (dp|ss) 13.7 -> 9.7; slower the classes at one wave per SIMD ((fp|ps)
// 30.6 -> 34.0, (dp|ps) 34.3 -> 38.0, (fs|ds) 22.7 -> 27.1, (pp|pp) 12.4 -> 14.6).
// Eight: the whole build 1103 -> 1230 ((ff|ps) 19.3 -> 53.6, (ps|ps) 57 -> 64).
template <int LI, int LJ, int LK, int LL> struct FourWaves { static constexpr bool ON = false; };
#define LANE_WAVES4(a, b, c, d) \
    template <> struct FourWaves<a, b, c, d> { static constexpr bool ON = true; };
LANE_WAVES4(1, 0, 0, 0) LANE_WAVES4(1, 0, 1, 0) LANE_WAVES4(1, 1, 0, 0) LANE_WAVES4(1, 1, 1, 0)
LANE_WAVES4(2, 0, 0, 0) LANE_WAVES4(2, 0, 1, 0) LANE_WAVES4(2, 0, 1, 1) LANE_WAVES4(2, 0, 2, 0)
LANE_WAVES4(2, 1, 0, 0) LANE_WAVES4(2, 2, 0, 0) LANE_WAVES4(3, 0, 0, 0) LANE_WAVES4(3, 0, 1, 0)
LANE_WAVES4(3, 1, 0, 0) LANE_WAVES4(3, 2, 1, 0) LANE_WAVES4(3, 3, 0, 0) LANE_WAVES4(3, 3, 1, 0)
#undef LANE_WAVES4

// Minimum waves per SIMD a class kernel is compiled for.  By default the
// compiler may use all 512 registers (one wave per SIMD); the classes below
// need a little over 256 and run faster with two waves per SIMD despite a few
// spilled registers (32-water def2-TZVP build, ms, one wave -> two:
// (fs|ps) 23.1 -> 16.9, (ds|pp) 15.2 -> 13.2, (ds|ds) 9.9 -> 7.1,
// (dd|pp) 11.6 -> 8.8, (fp|fp) 11.2 -> 8.5, (fd|dp) 9.4 -> 6.2; the classes
// that need 350 or more registers ran slower with two waves).  One wave per
// SIMD more for the smallest classes ((ss|ss) 6, (ps|ss) 5, (ps|ps) and
// (ds|ss) 4, (pp|ss) and (ds|ps) 3) measured slower on the 64-water build
// ((ps|ss) 119.3 -> 143.7 ms, whole build 2197 -> 2249 ms on one stream).
template <int LI, int LJ, int LK, int LL> struct ClassOcc { static constexpr int W = 1; };
#define CLASS_OCC2(a, b, c, d) \
    template <> struct ClassOcc<a, b, c, d> { static constexpr int W = 2; };
CLASS_OCC2(3, 0, 1, 0) CLASS_OCC2(2, 0, 1, 1) CLASS_OCC2(2, 0, 2, 0)
CLASS_OCC2(3, 1, 3, 1) CLASS_OCC2(3, 2, 2, 1) CLASS_OCC2(2, 2, 1, 1)
CLASS_OCC2(2, 1, 2, 2) CLASS_OCC2(3, 3, 3, 0) CLASS_OCC2(2, 2, 2, 1)
CLASS_OCC2(3, 0, 3, 2) CLASS_OCC2(3, 1, 2, 2) CLASS_OCC2(3, 3, 2, 1)
CLASS_OCC2(3, 2, 3, 0)
#undef CLASS_OCC2


template <int LI, int LJ, int LK, int LL, int PM, int NW>
__global__ __launch_bounds__((NW * WAVE), (ClassOcc<LI, LJ, LK, LL>::W))
void jk_lane_kernel(JKBuildArgs a, TaskBatch batch)
{
    int kl_chunk, use_lds;
    const int item = select_task(a, batch, kl_chunk, use_lds);
    constexpr int NFI = ncart(LI), NFJ = ncart(LJ);
    constexpr int N = (LI + LJ + LK + LL) / 2 + 1;
    __shared__ uint32_t queue_all[NW][2][2 * WAVE];
    __shared__ __align__(16) double moment_buf[MomentRows<N>::SIZE];
    const lds_double *rows = (const lds_double *)moment_buf;
    const int lane = threadIdx.x & (WAVE - 1);
    const int wid = threadIdx.x / WAVE;
    uint32_t *queue64 = queue_all[wid][0];
    uint32_t *queue32 = queue_all[wid][1];
    const int nbas = a.nbas, nao = a.nao;
    select_replica(a);
    WorkItem wi = work_item(a, item, kl_chunk, use_lds);
    const uint32_t bas_ij = a.pairs_ij[wi.pij];
    const float q_ij = a.q_ij[wi.pij];
    const float kl_cutoff = a.cutoff - q_ij;
    if (a.q_kl[wi.kl0] + a.dm_penalty + Q_COND_MARGIN < kl_cutoff) return;
    ShellPair sp;
    load_shell_pair(sp, bas_ij, nbas, a.bas, a.env, a.ao_loc);
    // K rows of this work item accumulated in LDS (one density)
    extern __shared__ double kacc_dyn[];
    const KRows kr = make_krows(kacc_dyn, use_lds, NFI + NFJ, wi);
    if (kr.on) {
        krows_zero(kr, NFI + NFJ, threadIdx.x, NW * WAVE);
        krows_load_d(kr, NFI, NFJ, sp.i0, sp.j0, nao, a.dm, threadIdx.x, NW * WAVE);
    }
    load_moment_rows<N>(moment_buf, a.rys, threadIdx.x, NW * WAVE);
    __syncthreads();
    int qn64 = 0, qn32 = 0;
    unsigned long long nsurv = 0, nsurv32 = 0, hsum = 0;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    bool stop = false;
    for (int base = wi.kl0 + wid * WAVE; base < wi.kl1 || qn64 > 0 || qn32 > 0;
         base += NW * WAVE) {
        if (base < wi.kl1 && !stop) {
            int pkl = base + lane;
            bool keep = false, fail_margin = false, lowp = false;
            if (pkl < wi.kl1) {
                float q_kl = a.q_kl[pkl];
                fail_margin = q_kl + a.dm_penalty + Q_COND_MARGIN < kl_cutoff;
                float dmax;
                const uint32_t bkl = a.pairs_kl[pkl];
                keep = survives_dmax(q_kl, kl_cutoff, a.dm_penalty, bas_ij, bkl,
                                     sp.ish, sp.jsh, nbas, a.dm_cond, a.screen, dmax,
                                     a.swap_ijkl != 0, q_ij, a.cutoff);
                lowp = keep && (q_ij + q_kl + dmax < a.fp32_cut);
                // the quartets of the other precision belong to the other launch
                if (PM == 1 && lowp) keep = lowp = false;
                if (PM == 2 && !lowp) keep = false;
                if (a.quartet_hash && keep) hsum += task_mix(a, bas_ij, bkl);
            }
            const uint64_t m64 = __ballot(keep && !lowp);
            const uint64_t m32 = __ballot(lowp);
            if (keep && !lowp) queue64[qn64 + __popcll(m64 & lt_mask)] = pkl;
            if (lowp) queue32[qn32 + __popcll(m32 & lt_mask)] = pkl;
            qn64 += __popcll(m64);
            qn32 += __popcll(m32);
            nsurv += __popcll(m64) + __popcll(m32);
            nsurv32 += __popcll(m32);
            stop = __ballot(fail_margin) != 0;
            wave_sync();
        }
        const bool flush = (base + NW * WAVE >= wi.kl1) || stop;
        if (PM != 2 && (qn64 >= WAVE || (flush && qn64 > 0))) {
            const int nb = min(qn64, WAVE);
            if constexpr (PM != 2)
                lane_batch<LI, LJ, LK, LL, double>(a, sp, bas_ij, wi.pij, queue64, nb, lane,
                                                   lt_mask, kr, rows);
            wave_sync();
            uint32_t rest = (nb + lane < qn64) ? queue64[nb + lane] : 0u;
            wave_sync();
            if (nb + lane < qn64) queue64[lane] = rest;
            qn64 -= nb;
            wave_sync();
        }
        if (PM != 1 && (qn32 >= WAVE || (flush && qn32 > 0))) {
            const int nb = min(qn32, WAVE);
            if constexpr (PM != 1)
                lane_batch<LI, LJ, LK, LL, float>(a, sp, bas_ij, wi.pij, queue32, nb, lane,
                                                  lt_mask, kr, rows);
            wave_sync();
            uint32_t rest = (nb + lane < qn32) ? queue32[nb + lane] : 0u;
            wave_sync();
            if (nb + lane < qn32) queue32[lane] = rest;
            qn32 -= nb;
            wave_sync();
        }
        if (flush && qn64 == 0 && qn32 == 0) break;
    }
    if (kr.on) {
        __syncthreads();
        krows_flush(kr, NFI, NFJ, sp.i0, sp.j0, nao, a.vk, threadIdx.x, NW * WAVE);
    }
    if (lane == 0) {
        if (a.n_quartets && nsurv) atomicAdd(a.n_quartets, nsurv);
        if (a.n_quartets_fp32 && nsurv32) atomicAdd(a.n_quartets_fp32, nsurv32);
    }
    if (a.quartet_hash && hsum) atomicAdd(a.quartet_hash, hsum);
}

// ---------------------------------------------------------------- one or two densities
// Per-lane kernel of the FP64 builds of ND = 1 or 2 densities with J and K (WJ, WK), J
// only or K only: what jk_lane_kernel decides at run time -- which matrices,
// where K is accumulated, the number of densities -- is fixed here, with the K
// rows and the density rows of the work item in LDS (KR_DROWS), J_ij and D_ij
// of the item in LDS, and its primitive records in LDS.
// These kernels wait for memory more than they compute: the load counter of a
// wavefront drains in order, so a load issued after the J_kl atomics of a batch
// waits for them.  A batch therefore keeps its J_kl block in registers, and the
// next batch adds it once its own first loads have arrived; the primitive loop
// then reads LDS only (for a ket of one primitive pair).
// 48 waters (def2-TZVP), one stream, ms: (ps|ss) 65.8 -> 58.5,
// (dp|ps) 40.6 -> 34.3, (dp|ss) 17.0 -> 13.7, (ds|ss) 29.0 -> 24.5, (ds|ps) 38.9 -> 35.4;
// the whole build on four streams 1000 -> 952.
// ND densities share the integrals, each with its own rows in LDS; the kernels for
// any number keep their K rows in HBM (two densities of 8 waters 53.6 -> 36.1 ms,
// of 12 waters 143 -> 75).
// Chunked classes with an f shell stay on jk_lane_kernel: the J_kl block held
// over the chunks costs them more registers than the waits ((fp|fs) 20.8 -> 22.5,
// (fp|pp) 33.7 -> 34.5, (fp|ds) 29.4 -> 29.9).
template <int LI, int LJ, int LK, int LL, bool WJ>
struct LaneFast {
    static constexpr bool ON = !WJ || LI < 3 || LaneChunk<LI, LJ, LK, LL>::NCH == 1;
};

struct ItemLds {
    const lds_double *pij, *dij;    // D_ij and J_ij: ij_step doubles from density to density
    lds_double *jij;
    const lds_double *rows;
    int kr_step;                    // K and density rows, from density to density
};

template <int LI, int LJ, int LK, int LL, bool WJ, bool WK, int ND>
__device__ __forceinline__ void lane_batch_fast(const JKBuildArgs &a, const ShellPair &sp,
                                                int pkl, uint32_t sh, bool active, int lane,
                                                const KRows &kr, const ItemLds &it,
                                                double *pend, uint32_t &pend_off)
{
    constexpr int NFI = ncart(LI), NFJ = ncart(LJ), NFK = ncart(LK), NFL = ncart(LL);
    constexpr int CH = LaneChunk<LI, LJ, LK, LL>::CH;
    const int nao = a.nao;
    const int ksh = sh >> 16, lsh = sh & 0xffff;
    double fac_sym = a.scale;
    if (sp.ish == sp.jsh) fac_sym *= .5;
    if (ksh == lsh) fac_sym *= .5;
    if (sp.ish == ksh && sp.jsh == lsh) fac_sym *= .5;
    if (!active) fac_sym = 0.;
    const double *rk = a.env + a.bas[ksh * 8 + 7], *rl = a.env + a.bas[lsh * 8 + 7];
    const double rk3[3] = {rk[0], rk[1], rk[2]};
    const double rkl[3] = {rl[0] - rk[0], rl[1] - rk[1], rl[2] - rk[2]};
    const int nij = a.iprim * a.jprim, nkl = a.kprim * a.lprim;
    const int k0 = a.ao_loc[ksh], l0 = a.ao_loc[lsh];
    // columns of this quartet's k and l AOs in the LDS rows
    const int dk = k0 - kr.k_ao0, dl = kr.loff + l0 - kr.l_ao0;
    const uint32_t off_kl = (uint32_t)k0 * (uint32_t)nao + (uint32_t)l0;
    constexpr int NFKL = NFK * NFL;
    double vkl[ND * NFKL];
#pragma unroll
    for (int n = 0; n < ND * NFKL; ++n) vkl[n] = 0.;
    lane_chunks<(NFI + CH - 1) / CH>([&](auto cc) {
        constexpr int I0 = decltype(cc)::value * CH;
        constexpr int I1 = I0 + CH < NFI ? I0 + CH : NFI;
        constexpr int NI = I1 - I0;
        double gout[NI * NFJ * NFK * NFL];
        eri_lane<LI, LJ, LK, LL, double, I0, I1, !WJ>(
            gout, PijLds{it.pij}, nij, a.pdata_kl + (size_t)pkl * nkl * PREC, nkl, sp.rij, rk3,
            rkl, a.rys, it.rows, fac_sym, Oper<!WJ>(a), [&] {
                if constexpr (WJ && I0 == 0) {
                    // J_kl of the previous batch
                    if (pend_off != ~0u) {
#pragma unroll
                        for (int id = 0; id < ND; ++id) {
                            double *J = a.vj + (size_t)id * nao * nao + pend_off;
#pragma unroll
                            for (int n = 0; n < NFKL; ++n)
                                atomic_add(J + (uint32_t)((n / NFL) * nao + n % NFL),
                                           pend[id * NFKL + n]);
                        }
                    }
                }
            });
#pragma unroll
        for (int id = 0; id < ND; ++id) {
            lds_double *kp = kr.p + id * it.kr_step;
            const lds_double *kd = kr.d + id * it.kr_step;
            if constexpr (WK) {
                // K_ik += (ij|kl) D_jl ; K_il += (ij|kl) D_jk
#pragma unroll
                for (int i = I0; i < I1; ++i) {
                    double kil[NFL], kik[NFK];
#pragma unroll
                    for (int l = 0; l < NFL; ++l) kil[l] = 0.;
#pragma unroll
                    for (int k = 0; k < NFK; ++k) kik[k] = 0.;
                    if (active) {
#pragma unroll
                        for (int j = 0; j < NFJ; ++j) {
                            const lds_double *dj = kd + (NFI + j) * kr.width;
#pragma unroll
                            for (int k = 0; k < NFK; ++k)
#pragma unroll
                            for (int l = 0; l < NFL; ++l) {
                                const double g = gout[(((i - I0)*NFJ + j)*NFK + k)*NFL + l];
                                kil[l] = fma(g, dj[dk + k], kil[l]);
                                kik[k] = fma(g, dj[dl + l], kik[k]);
                            }
                        }
#pragma unroll
                        for (int k = 0; k < NFK; ++k) lds_add(kp + i * kr.width + dk + k, kik[k]);
#pragma unroll
                        for (int l = 0; l < NFL; ++l) lds_add(kp + i * kr.width + dl + l, kil[l]);
                    }
                }
                // K_jk += (ij|kl) D_il ; K_jl += (ij|kl) D_ik
#pragma unroll
                for (int j = 0; j < NFJ; ++j) {
                    double kjl[NFL], kjk[NFK];
#pragma unroll
                    for (int l = 0; l < NFL; ++l) kjl[l] = 0.;
#pragma unroll
                    for (int k = 0; k < NFK; ++k) kjk[k] = 0.;
                    if (active) {
#pragma unroll
                        for (int i = I0; i < I1; ++i) {
                            const lds_double *di = kd + i * kr.width;
#pragma unroll
                            for (int k = 0; k < NFK; ++k)
#pragma unroll
                            for (int l = 0; l < NFL; ++l) {
                                const double g = gout[(((i - I0)*NFJ + j)*NFK + k)*NFL + l];
                                kjl[l] = fma(g, di[dk + k], kjl[l]);
                                kjk[k] = fma(g, di[dl + l], kjk[k]);
                            }
                        }
                        lds_double *kj = kp + (NFI + j) * kr.width;
#pragma unroll
                        for (int k = 0; k < NFK; ++k) lds_add(kj + dk + k, kjk[k]);
#pragma unroll
                        for (int l = 0; l < NFL; ++l) lds_add(kj + dl + l, kjl[l]);
                    }
                }
            }
            if constexpr (WJ) {
                double dkl[NFKL];
                const double *D = a.dm + (size_t)id * nao * nao + off_kl;
#pragma unroll
                for (int n = 0; n < NFKL; ++n) dkl[n] = D[(uint32_t)((n / NFL) * nao + n % NFL)];
                double vij[NI * NFJ];
#pragma unroll
                for (int i = I0; i < I1; ++i)
#pragma unroll
                for (int j = 0; j < NFJ; ++j) {
                    const double d = it.dij[2 * id * NFI * NFJ + i * NFJ + j];
                    double s = 0.;
#pragma unroll
                    for (int n = 0; n < NFKL; ++n) {
                        const double g = gout[((i - I0)*NFJ + j)*NFKL + n];
                        s = fma(g, dkl[n], s);
                        vkl[id * NFKL + n] = fma(g, d, vkl[id * NFKL + n]);
                    }
                    // (an inactive lane's integrals are zero)
                    vij[(i - I0)*NFJ + j] = s;
                }
                wave_reduce_scatter<NI * NFJ>(vij, lane, [&](int n, double x) {
                    lds_add(it.jij + 2 * id * NFI * NFJ + I0 * NFJ + n, x);
                });
            }
        }
    });
    if constexpr (WJ) {
#pragma unroll
        for (int n = 0; n < ND * NFKL; ++n) pend[n] = vkl[n];
        pend_off = active ? off_kl : ~0u;
    }
}

template <int LI, int LJ, int LK, int LL, bool WJ, bool WK, int NW, int ND>
__global__ __launch_bounds__((NW * WAVE), (ClassOcc<LI, LJ, LK, LL>::W))
void jk_lane_fast_kernel(JKBuildArgs a, TaskBatch batch)
{
    int kl_chunk, use_lds, dm0;
    const int item = select_task(a, batch, kl_chunk, use_lds, dm0);
    constexpr int NFI = ncart(LI), NFJ = ncart(LJ), NFKL = ncart(LK) * ncart(LL);
    constexpr int N = (LI + LJ + LK + LL) / 2 + 1;
    constexpr int NT = NW * WAVE;
    __shared__ uint32_t queue_all[NW][2][2 * WAVE];
    __shared__ int left[NW];
    __shared__ __align__(16) double moment_buf[MomentRows<N>::SIZE];
    __shared__ double ij_buf[2 * ND][NFI * NFJ];
    extern __shared__ __align__(16) double fast_dyn[];
    const int tid = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int wid = tid / WAVE;
    uint32_t *queue = queue_all[wid][0], *queue_sh = queue_all[wid][1];
    const int nbas = a.nbas, nao = a.nao;
    select_replica(a);
    const size_t nao2 = (size_t)nao * nao;
    a.dm += dm0 * nao2;
    if constexpr (WJ) a.vj += dm0 * nao2;
    if constexpr (WK) a.vk += dm0 * nao2;
    const WorkItem wi = work_item(a, item, kl_chunk, use_lds);
    const uint32_t bas_ij = a.pairs_ij[wi.pij];
    const float q_ij = a.q_ij[wi.pij];
    const float kl_cutoff = a.cutoff - q_ij;
    if (a.q_kl[wi.kl0] + a.dm_penalty + Q_COND_MARGIN < kl_cutoff) return;
    ShellPair sp;
    load_shell_pair(sp, bas_ij, nbas, a.bas, a.env, a.ao_loc);
    const float dc_ij = a.dm_cond[bas_ij];
    const int nij = a.iprim * a.jprim;
    // LDS: primitive records of ij, then the K rows and the density rows
    ItemLds it;
    lds_double *pij = (lds_double *)fast_dyn;
    it.pij = pij;
    it.dij = (lds_double *)ij_buf[0];
    it.jij = (lds_double *)ij_buf[1];
    it.rows = (lds_double *)moment_buf;
    const KRows kr = make_krows(fast_dyn + nij * PIJ_LDS, WK ? 2 | KR_DROWS : 0, NFI + NFJ, wi);
    it.kr_step = 2 * (NFI + NFJ) * kr.width;
    if constexpr (WK) {
#pragma unroll
        for (int id = 0; id < ND; ++id) {
            const KRows krd = krows_of(kr, id * it.kr_step);
            krows_zero(krd, NFI + NFJ, tid, NT);
            krows_load_d(krd, NFI, NFJ, sp.i0, sp.j0, nao, a.dm + id * nao2, tid, NT);
        }
    }
    stage_pij(pij, a.pdata_ij + (size_t)wi.pij * nij * PREC, nij, sp.ri, tid, NT);
    load_moment_rows<N>(moment_buf, a.rys, tid, NT);
    for (int n = tid; n < NFI * NFJ; n += NT) {
#pragma unroll
        for (int id = 0; id < ND; ++id) {
            ij_buf[2 * id][n] = a.dm[id * nao2 + (size_t)(sp.i0 + n / NFJ) * nao + sp.j0 + n % NFJ];
            ij_buf[2 * id + 1][n] = 0.;
        }
    }
    __syncthreads();
    int qn = 0;
    unsigned long long nsurv = 0, hsum = 0;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    double pend[WJ ? ND * NFKL : 1];
    uint32_t pend_off = ~0u;
#pragma unroll
    for (int n = 0; n < (WJ ? ND * NFKL : 1); ++n) pend[n] = 0.;
    // floor(b / nbas) of a pair id: the reciprocal's estimate is at most one
    // too large
    const uint32_t nbas_inv = 0xffffffffu / (uint32_t)nbas + 1u;
    bool stop = false;
    int base = wi.kl0 + wid * WAVE;
    bool last = false;
    while (!last) {
        // survivors until a batch is full
        while (qn < WAVE && base < wi.kl1 && !stop) {
            const int pkl = base + lane;
            bool keep = false, fail_margin = false;
            uint32_t sh = 0;
            if (pkl < wi.kl1) {
                const float q_kl = a.q_kl[pkl];
                const uint32_t bkl = a.pairs_kl[pkl];
                fail_margin = q_kl + a.dm_penalty + Q_COND_MARGIN < kl_cutoff;
                uint32_t ksh = nbas > 1 ? __umulhi(bkl, nbas_inv) : bkl;
                if (ksh * (uint32_t)nbas > bkl) --ksh;
                const uint32_t lsh = bkl - ksh * (uint32_t)nbas;
                sh = ksh << 16 | lsh;
                keep = survives_sh(q_kl, kl_cutoff, a.dm_penalty, bas_ij, bkl, sp.ish, sp.jsh,
                                   (int)ksh, (int)lsh, nbas, a.dm_cond, dc_ij, a.screen,
                                   a.swap_ijkl != 0, q_ij, a.cutoff);
                if (a.quartet_hash && keep) hsum += task_mix(a, bas_ij, bkl);
            }
            const uint64_t m = __ballot(keep);
            if (keep) {
                const int n = qn + __popcll(m & lt_mask);
                queue[n] = pkl;
                queue_sh[n] = sh;
            }
            qn += __popcll(m);
            nsurv += __popcll(m);
            stop = __ballot(fail_margin) != 0;
            wave_sync();
            base += NT;
        }
        // the newest WAVE entries of the queue; at the end the wavefronts'
        // remainders together, one batch each
        int w = wid, n = qn - WAVE + lane;
        bool active = true;
        if (qn >= WAVE) {
            qn -= WAVE;
        } else {
            if (lane == 0) left[wid] = qn;
            __syncthreads();
            int total = 0;
#pragma unroll
            for (int v = 0; v < NW; ++v) total += left[v];
            if (wid * WAVE >= total) break;
            active = wid * WAVE + lane < total;
            n = active ? wid * WAVE + lane : 0;
            for (w = 0; n >= left[w]; ++w) n -= left[w];
            last = true;
        }
        lane_batch_fast<LI, LJ, LK, LL, WJ, WK, ND>(a, sp, queue_all[w][0][n], queue_all[w][1][n],
                                                    active, lane, kr, it, pend, pend_off);
        wave_sync();
    }
    if constexpr (WJ) {
        if (pend_off != ~0u) {
            constexpr int NFL = ncart(LL);
#pragma unroll
            for (int n = 0; n < ND * NFKL; ++n)
                atomic_add(a.vj + (n / NFKL) * nao2 + pend_off +
                               (uint32_t)((n % NFKL / NFL) * nao + n % NFL), pend[n]);
        }
    }
    __syncthreads();
    if constexpr (WK) {
#pragma unroll
        for (int id = 0; id < ND; ++id)
            krows_flush(krows_of(kr, id * it.kr_step), NFI, NFJ, sp.i0, sp.j0, nao,
                        a.vk + id * nao2, tid, NT);
    }
    if constexpr (WJ) {
#pragma unroll
        for (int id = 0; id < ND; ++id)
            for (int n = tid; n < NFI * NFJ; n += NT)
                atomic_add(a.vj + id * nao2 + (size_t)(sp.i0 + n / NFJ) * nao + sp.j0 + n % NFJ,
                           ij_buf[2 * id + 1][n]);
    }
    if (lane == 0 && a.n_quartets && nsurv) atomicAdd(a.n_quartets, nsurv);
    if (a.quartet_hash && hsum) atomicAdd(a.quartet_hash, hsum);
}

// ---------------------------------------------------------------- team
// Team of TS lanes per quartet, NQ quartets per block of TB threads.
template <int LI, int LJ, int LK, int LL>
struct TeamShape {
    static constexpr int NFI = ncart(LI), NFJ = ncart(LJ), NFK = ncart(LK), NFL = ncart(LL);
    static constexpr int NROWS = NFI * NFJ;
    static constexpr int NFKL = NFK * NFL;
    static constexpr int N = (LI + LJ + LK + LL) / 2 + 1;
    static constexpr int GS = (LI+1)*(LJ+1)*(LK+1)*(LL+1);
    static constexpr int TS0 = NROWS > 3 * N ? NROWS : 3 * N;
    static constexpr int TB1 = TS0 <= 64 ? 64 : (TS0 <= 128 ? 128 : 256);
    static constexpr int TB = TB1 < TEAM_TB_MIN ? TEAM_TB_MIN : TB1;
    static constexpr int G_DBL = 2 * N + N * 3 * GS;            // roots + 2D integrals
    static constexpr int S_ROWS0 = 4096 / NFKL;                 // rows staged per pass
    static constexpr int S_ROWS = S_ROWS0 < NROWS ? (S_ROWS0 > 0 ? S_ROWS0 : 1) : NROWS;
    static constexpr int S_DBL = S_ROWS * NFKL;
    static constexpr int PER_Q = G_DBL > S_DBL ? G_DBL : S_DBL;
    static constexpr int NQ0 = TB / TS0;
    static constexpr int NQ1 = (6144 / PER_Q) > 0 ? (6144 / PER_Q) : 1;   // 48 KB of LDS
    static constexpr int NQ = NQ0 < NQ1 ? NQ0 : NQ1;
    static constexpr int TS = TB / NQ;
    // primitive quartets per pass: the 3N lanes of one primitive quartet's
    // 2D tables are replicated PB times over the team, within the same
    // 48 KB of LDS (one pass of roots, tables and triple products, three
    // block barriers, per PB primitive quartets)
    static constexpr int PB_LANES = TS / (3 * N) > 0 ? TS / (3 * N) : 1;
    static constexpr int PB_LDS0 = 6144 / (NQ * G_DBL);
    static constexpr int PB_LDS = PB_LDS0 > 0 ? PB_LDS0 : 1;
    static constexpr int PB = TEAM_PRIM_BATCH ? (PB_LANES < PB_LDS ? PB_LANES : PB_LDS) : 1;
    static constexpr int G_ALL = PB * G_DBL;
    static constexpr int PER_QB = G_ALL > S_DBL ? G_ALL : S_DBL;
    // per-team staging of the density blocks of the current quartet:
    // D_kl, then rows r of i (r < NFI) and j with their k and l columns,
    // then D_ij (used when several densities are digested)
    static constexpr int DROW = NFK + NFL;
    static constexpr int D_KL = 0, D_R = NFKL, D_IJ = D_R + (NFI + NFJ) * DROW;
    static constexpr int DSZ = D_IJ + NFI * NFJ;
};

template <int LI, int LJ, int LK, int LL>
__global__ __launch_bounds__((TeamShape<LI, LJ, LK, LL>::TB),
                             (TEAM_MIN_WAVES > ClassOcc<LI, LJ, LK, LL>::W ?
                              TEAM_MIN_WAVES : ClassOcc<LI, LJ, LK, LL>::W))
void jk_team_kernel(JKBuildArgs a, TaskBatch batch)
{
    int kl_chunk, use_lds;
    const int item = select_task(a, batch, kl_chunk, use_lds);
    using S = TeamShape<LI, LJ, LK, LL>;
    constexpr int NFI = S::NFI, NFJ = S::NFJ, NFK = S::NFK, NFL = S::NFL;
    constexpr int NROWS = S::NROWS, NFKL = S::NFKL, N = S::N, GS = S::GS;
    constexpr int TB = S::TB, NQ = S::NQ, TS = S::TS;
    constexpr int NW = TB / WAVE;
    constexpr CartPow<LI> ci{};
    constexpr CartPow<LJ> cj{};
    constexpr CartPow<LK> ck{};
    constexpr CartPow<LL> cl{};
    constexpr int SJ = LL+1, SK = (LK+1)*(LL+1), SI = (LJ+1)*(LK+1)*(LL+1);

    __shared__ uint32_t queue[2 * TB];
    __shared__ int wave_cnt[NW + 1];
    __shared__ int stop_flag;
    __shared__ double lds[NQ * S::PER_QB];
    __shared__ double dstage[NQ * S::DSZ];
    __shared__ double dij_blk[NFI * NFJ];     // D_ij of the work item (one density)

    const int tid = threadIdx.x;
    const int lane = tid & (WAVE - 1);
    const int wid = tid / WAVE;
    const int team = tid / TS;
    const int tl = tid - team * TS;
    const int nbas = a.nbas, nao = a.nao;
    const size_t nao2 = (size_t)nao * nao;
    select_replica(a);
    WorkItem wi = work_item(a, item, kl_chunk, use_lds);
    const uint32_t bas_ij = a.pairs_ij[wi.pij];
    const float kl_cutoff = a.cutoff - a.q_ij[wi.pij];
    if (a.q_kl[wi.kl0] + a.dm_penalty + Q_COND_MARGIN < kl_cutoff) return;
    ShellPair sp;
    load_shell_pair(sp, bas_ij, nbas, a.bas, a.env, a.ao_loc);
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    constexpr int PB = S::PB;
    double *my = lds + (team < NQ ? team : 0) * S::PER_QB;
    // per primitive quartet p < PB of a pass: roots and weights at
    // my + p * G_DBL ([2N]), then its 2D tables ([N][3][GS])
    const int row = tl;               // (i, j) row owned by this lane
    const bool has_row = team < NQ && row < NROWS;
    const int irow = has_row ? row / NFJ : 0, jrow = has_row ? row % NFJ : 0;
    // J_ij of this lane's row, summed over the block's quartets (one density)
    double vj_row = 0.;
    // K rows of this work item accumulated in LDS (one density)
    extern __shared__ double kacc_dyn[];
    const KRows kr = make_krows(kacc_dyn, use_lds, NFI + NFJ, wi);
    krows_zero(kr, NFI + NFJ, tid, TB);
    for (int n = tid; n < NFI * NFJ; n += TB)
        dij_blk[n] = a.dm[(size_t)(sp.i0 + n / NFJ) * nao + sp.j0 + n % NFJ];
    double *dsh = dstage + (team < NQ ? team : 0) * S::DSZ;
    __syncthreads();
    int qn = 0;
    unsigned long long nsurv = 0, hsum = 0;
    bool stop = false;
    for (int base = wi.kl0; ; base += TB) {
        if (base < wi.kl1 && !stop) {
            int pkl = base + tid;
            bool keep = false, fail_margin = false;
            uint32_t bkl = 0;
            if (pkl < wi.kl1) {
                float q_kl = a.q_kl[pkl];
                bkl = a.pairs_kl[pkl];
                fail_margin = q_kl + a.dm_penalty + Q_COND_MARGIN < kl_cutoff;
                keep = survives(q_kl, kl_cutoff, a.dm_penalty, bas_ij, bkl,
                                sp.ish, sp.jsh, nbas, a.dm_cond, a.screen, a.swap_ijkl != 0,
                                a.q_ij[wi.pij], a.cutoff);
                if (a.quartet_hash && keep) hsum += task_mix(a, bas_ij, bkl);
            }
            uint64_t m = __ballot(keep);
            uint64_t mf = __ballot(fail_margin);
            if (tid == 0) stop_flag = 0;
            __syncthreads();
            if (lane == 0) {
                wave_cnt[wid] = __popcll(m);
                if (mf) stop_flag = 1;
            }
            __syncthreads();
            int off = qn;
            for (int w = 0; w < wid; ++w) off += wave_cnt[w];
            if (keep) queue[off + __popcll(m & lt_mask)] = pkl;
            int tot = 0;
            for (int w = 0; w < NW; ++w) tot += wave_cnt[w];
            qn += tot;
            nsurv += tot;
            stop = stop_flag != 0;
            __syncthreads();
        }
        bool flush = base + TB >= wi.kl1 || stop;
        int head = 0;
        while (qn - head >= NQ || (flush && head < qn)) {
            // team `team` evaluates queue[head + team]
            const int qidx = head + team;
            const bool active = team < NQ && qidx < qn;
            const int pkl = queue[active ? qidx : head];
            uint32_t bas_kl = a.pairs_kl[pkl];
            int ksh = bas_kl / nbas, lsh = bas_kl - (bas_kl / nbas) * nbas;
            double fac_sym = a.scale;
            if (sp.ish == sp.jsh) fac_sym *= .5;
            if (ksh == lsh) fac_sym *= .5;
            if (bas_ij == bas_kl) fac_sym *= .5;
            const double *rk = a.env + a.bas[ksh * 8 + 7], *rl = a.env + a.bas[lsh * 8 + 7];
            double rkl[3] = {rl[0] - rk[0], rl[1] - rk[1], rl[2] - rk[2]};
            const Oper<true> op(a);
            const int nij = a.iprim * a.jprim, nkl = a.kprim * a.lprim;
            const double *pdij = a.pdata_ij + (size_t)wi.pij * nij * PREC;
            const double *pdkl = a.pdata_kl + (size_t)pkl * nkl * PREC;
            double acc[NFKL];
#pragma unroll
            for (int n = 0; n < NFKL; ++n) acc[n] = 0.;
            const int npq = nij * nkl;
            // primitive-pair quantities of primitive quartet pq (ij fastest)
            auto prim = [&](int pq, double &aij, double &raij, double &akl, double &rakl,
                            double *PA, double *PQ, double *QC, double &r_aa, double &theta,
                            double &rr, double &fac) {
                const int kp = pq / nij, ip = pq - kp * nij;
                const double *qr = pdkl + kp * PREC;
                const double *pr = pdij + ip * PREC;
                akl = qr[0]; rakl = qr[1];
                aij = pr[0]; raij = pr[1];
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    PA[d] = pr[2+d] - sp.ri[d];
                    PQ[d] = pr[2+d] - qr[2+d];
                    QC[d] = qr[2+d] - rk[d];
                }
                rr = PQ[0]*PQ[0] + PQ[1]*PQ[1] + PQ[2]*PQ[2];
                r_aa = 1. / (aij + akl);
                theta = aij * akl * r_aa;
                fac = pr[5] * qr[5] * fac_sym * sqrt(r_aa);
            };
#pragma unroll 1
            for (int part = op.parts() - 1; part >= 0; --part) {
            const double omega2 = part ? 0. : op.omega2;
                for (int pq0 = 0; pq0 < npq; pq0 += PB) {
                    const int np = min(PB, npq - pq0);
                    __syncthreads();
                    // roots: lane (p, r) for p < np, r < N
                    if (active && tl < np * N) {
                        const int p = tl / N, r = tl - p * N;
                        double aij, raij, akl, rakl, PA[3], PQ[3], QC[3], r_aa, theta, rr, fac;
                        prim(pq0 + p, aij, raij, akl, rakl, PA, PQ, QC, r_aa, theta, rr, fac);
                        double rt, wt;
                        if (omega2 > 0.) {
                            // long-range attenuation (see eri_lane)
                            const double aw = omega2 / (omega2 + theta);
                            rys_root_one<N>(a.rys, theta * rr * aw, r, rt, wt);
                            rt *= aw; wt *= sqrt(aw);
                        } else {
                            rys_root_one<N>(a.rys, theta * rr, r, rt, wt);
                        }
                        double *rw = my + p * S::G_DBL;
                        rw[2*r] = rt; rw[2*r+1] = wt;
                    }
                    __syncthreads();
                    // 2D tables: lane (p, r, d) for p < np
                    if (active && tl < np * 3 * N) {
                        const int p = tl / (3 * N), rd = tl - p * (3 * N);
                        const int r = rd / 3, d = rd - (rd / 3) * 3;
                        double aij, raij, akl, rakl, PA[3], PQ[3], QC[3], r_aa, theta, rr, fac;
                        prim(pq0 + p, aij, raij, akl, rakl, PA, PQ, QC, r_aa, theta, rr, fac);
                        const double *rw = my + p * S::G_DBL;
                        double rt_aa = rw[2*r] * r_aa;
                        double rt_aij = rt_aa * akl, rt_akl = rt_aa * aij;
                        double b10 = .5 * raij * (1. - rt_aij);
                        double b01 = .5 * rakl * (1. - rt_akl);
                        double b00 = .5 * rt_aa;
                        double g[GS];
                        double pa = d == 0 ? PA[0] : (d == 1 ? PA[1] : PA[2]);
                        double pq = d == 0 ? PQ[0] : (d == 1 ? PQ[1] : PQ[2]);
                        double qc = d == 0 ? QC[0] : (d == 1 ? QC[1] : QC[2]);
                        double rd_ = d == 0 ? sp.rij[0] : (d == 1 ? sp.rij[1] : sp.rij[2]);
                        double kd = d == 0 ? rkl[0] : (d == 1 ? rkl[1] : rkl[2]);
                        double g00 = d == 2 ? rw[2*r+1] * (part ? fac * op.full : fac) : 1.;
                        build_g<LI, LJ, LK, LL, double>(g, g00, pa - rt_aij * pq,
                                                qc + rt_akl * pq,
                                                b10, b01, b00, rd_, kd);
                        double *dst = my + p * S::G_DBL + 2 * N + (r * 3 + d) * GS;
#pragma unroll
                        for (int n = 0; n < GS; ++n) dst[n] = g[n];
                    }
                    __syncthreads();
                    if (active && has_row) {
                        int ax = 0, ay = 0, az = 0, bx = 0, by = 0, bz = 0;
                        // Cartesian powers of this row's i and j (runtime lookup)
#pragma unroll
                        for (int i = 0; i < NFI; ++i)
                            if (i == irow) { ax = ci.x[i]; ay = ci.y[i]; az = ci.z[i]; }
#pragma unroll
                        for (int j = 0; j < NFJ; ++j)
                            if (j == jrow) { bx = cj.x[j]; by = cj.y[j]; bz = cj.z[j]; }
                        const int ox = ax * SI + bx * SK, oy = ay * SI + by * SK, oz = az * SI + bz * SK;
                        for (int p = 0; p < np; ++p) {
                            const double *gb = my + p * S::G_DBL + 2 * N;
                            for (int r = 0; r < N; ++r) {
                                const double *gx = gb + (r * 3 + 0) * GS + ox;
                                const double *gy = gb + (r * 3 + 1) * GS + oy;
                                const double *gz = gb + (r * 3 + 2) * GS + oz;
                                double sx[SK], sy[SK], sz[SK];
#pragma unroll
                                for (int n = 0; n < SK; ++n) { sx[n] = gx[n]; sy[n] = gy[n]; sz[n] = gz[n]; }
#pragma unroll
                                for (int k = 0; k < NFK; ++k)
#pragma unroll
                                for (int l = 0; l < NFL; ++l) {
                                    int kx = ck.x[k]*SJ + cl.x[l];
                                    int ky = ck.y[k]*SJ + cl.y[l];
                                    int kz = ck.z[k]*SJ + cl.z[l];
                                    acc[k*NFL + l] = fma(sx[kx] * sy[ky], sz[kz], acc[k*NFL + l]);
                                }
                            }
                        }
                    }
                }
            }
            // ---- digestion of the team's quartet
            const int i0 = sp.i0, j0 = sp.j0;
            const int k0 = a.ao_loc[ksh], l0 = a.ao_loc[lsh];
            double *stage = my;       // reuse the team's LDS
            constexpr int DROW = S::DROW;
            const double *dkl = dsh + S::D_KL, *drow = dsh + S::D_R;
            for (int id = 0; id < a.n_dm; ++id) {
                const double *D = a.dm + id * nao2;
                // the quartet's density blocks into the team's LDS, one
                // cooperative gather
                __syncthreads();
                if (active) {
                    for (int n = tl; n < S::DSZ; n += TS) {
                        size_t idx;
                        if (n < S::D_R) {
                            idx = (size_t)(k0 + n / NFL) * nao + l0 + n % NFL;
                        } else if (n < S::D_IJ) {
                            const int r = (n - S::D_R) / DROW, c = (n - S::D_R) - r * DROW;
                            const int ao = r < NFI ? i0 + r : j0 + r - NFI;
                            idx = (size_t)ao * nao + (c < NFK ? k0 + c : l0 + c - NFK);
                        } else {
                            if (a.n_dm == 1) continue;
                            const int m = n - S::D_IJ;
                            idx = (size_t)(i0 + m / NFJ) * nao + j0 + m % NFJ;
                        }
                        dsh[n] = D[idx];
                    }
                }
                __syncthreads();
                const double *dij = a.n_dm == 1 ? dij_blk : dsh + S::D_IJ;
                if (a.vj && active && has_row) {
                    double s = 0.;
#pragma unroll
                    for (int k = 0; k < NFK; ++k)
#pragma unroll
                    for (int l = 0; l < NFL; ++l)
                        s = fma(acc[k*NFL + l], dkl[k*NFL + l], s);
                    if (a.n_dm == 1) vj_row += s;
                    else atomic_add(a.vj + id * nao2 + (i0+irow)*nao + j0+jrow, s);
                }
                for (int r0 = 0; r0 < NROWS; r0 += S::S_ROWS) {
                    const int r1 = min(r0 + S::S_ROWS, NROWS);
                    __syncthreads();
                    if (active && has_row && row >= r0 && row < r1) {
#pragma unroll
                        for (int n = 0; n < NFKL; ++n) stage[(row - r0) * NFKL + n] = acc[n];
                    }
                    __syncthreads();
                    if (!active) continue;
                    if (a.vj) {
                        double *J = a.vj + id * nao2;
                        for (int e = tl; e < NFKL; e += TS) {
                            int k = e / NFL, l = e - (e / NFL) * NFL;
                            double s = 0.;
                            for (int rr = r0; rr < r1; ++rr)
                                s = fma(stage[(rr - r0) * NFKL + e], dij[rr], s);
                            atomic_add(J + (k0+k)*nao + l0+l, s);
                        }
                    }
                    if (a.vk) {
                        double *K = a.vk + id * nao2;
                        const int ilo = r0 / NFJ, ihi = (r1 - 1) / NFJ;
                        const int ni = ihi - ilo + 1;
                        // K_ik (sum over j,l of D_jl) and K_il (sum over j,k of D_jk)
                        for (int e = tl; e < ni * (NFK + NFL); e += TS) {
                            int i = ilo + e / (NFK + NFL);
                            int m = e - (e / (NFK + NFL)) * (NFK + NFL);
                            double s = 0.;
                            for (int j = 0; j < NFJ; ++j) {
                                int rr = i * NFJ + j;
                                if (rr < r0 || rr >= r1) continue;
                                const double *srow = stage + (rr - r0) * NFKL;
                                const double *dj = drow + (NFI + j) * DROW;
                                if (m < NFK) {
                                    for (int l = 0; l < NFL; ++l)
                                        s = fma(srow[m*NFL + l], dj[NFK + l], s);
                                } else {
                                    int l = m - NFK;
                                    for (int k = 0; k < NFK; ++k)
                                        s = fma(srow[k*NFL + l], dj[k], s);
                                }
                            }
                            if (m < NFK) {
                                if (kr.kcols) lds_add(kr.p + i * kr.width + k0 + m - kr.k_ao0, s);
                                else atomic_add(K + (i0+i)*nao + k0+m, s);
                            } else if (kr.on) {
                                lds_add(kr.p + i * kr.width + kr.loff + l0 + m - NFK - kr.l_ao0, s);
                            } else {
                                atomic_add(K + (i0+i)*nao + l0+m-NFK, s);
                            }
                        }
                        // K_jk (sum over i,l of D_il) and K_jl (sum over i,k of D_ik)
                        for (int e = tl; e < NFJ * (NFK + NFL); e += TS) {
                            int j = e / (NFK + NFL);
                            int m = e - j * (NFK + NFL);
                            double s = 0.;
                            for (int i = ilo; i <= ihi; ++i) {
                                int rr = i * NFJ + j;
                                if (rr < r0 || rr >= r1) continue;
                                const double *srow = stage + (rr - r0) * NFKL;
                                const double *di = drow + i * DROW;
                                if (m < NFK) {
                                    for (int l = 0; l < NFL; ++l)
                                        s = fma(srow[m*NFL + l], di[NFK + l], s);
                                } else {
                                    int l = m - NFK;
                                    for (int k = 0; k < NFK; ++k)
                                        s = fma(srow[k*NFL + l], di[k], s);
                                }
                            }
                            if (m < NFK) {
                                if (kr.kcols) lds_add(kr.p + (NFI + j) * kr.width + k0 + m - kr.k_ao0, s);
                                else atomic_add(K + (j0+j)*nao + k0+m, s);
                            } else if (kr.on) {
                                lds_add(kr.p + (NFI + j) * kr.width + kr.loff + l0 + m - NFK - kr.l_ao0, s);
                            } else {
                                atomic_add(K + (j0+j)*nao + l0+m-NFK, s);
                            }
                        }
                    }
                }
            }
            __syncthreads();
            head += NQ;
        }
        // move the unprocessed remainder to the front of the queue
        int rem = qn - head;
        uint32_t v = 0;
        if (tid < rem) v = queue[head + tid];
        __syncthreads();
        if (tid < rem) queue[tid] = v;
        qn = rem;
        __syncthreads();
        if (flush) break;
    }
    if (a.vj && a.n_dm == 1 && has_row && vj_row != 0.)
        atomic_add(a.vj + (sp.i0 + irow)*nao + sp.j0 + jrow, vj_row);
    if (kr.on) {
        __syncthreads();
        krows_flush(kr, NFI, NFJ, sp.i0, sp.j0, nao, a.vk, tid, TB);
    }
    if (a.n_quartets && tid == 0 && nsurv) atomicAdd(a.n_quartets, nsurv);
    if (a.quartet_hash && hsum) atomicAdd(a.quartet_hash, hsum);
}

// ---------------------------------------------------------------- class info
template <int LI, int LJ, int LK, int LL>
struct ClassTraits {
    static constexpr int NF = ncart(LI) * ncart(LJ) * ncart(LK) * ncart(LL);
    static constexpr int GS = (LI+1)*(LJ+1)*(LK+1)*(LL+1);
    static constexpr int N = (LI + LJ + LK + LL) / 2 + 1;
    // per-lane path when the block and three 2D tables fit in LANE_MAX doubles,
    // or when chunks of at most LANE_MAX_CHUNKS row blocks of the block do
    static constexpr bool LANE = (NF + 3 * GS <= LANE_MAX ||
                                  (LaneChunk<LI, LJ, LK, LL>::FIT > 0 &&
                                   (LaneChunked<LI, LJ, LK, LL>::ON ||
                                    LaneChunk<LI, LJ, LK, LL>::NCH <= LANE_MAX_CHUNKS))) &&
                                 NF != LANE_SKIP_NF;
};

// What the launcher (jk_launch.hip) needs to know of one class's kernel.
#define JK_MAX_DEVICES 64
#define JK_FAST 2
#define JK_FOUR 5
#define JK_TWO 8
#define JK_KERNELS 13
// wavefronts of kernel n of the per-lane classes, and densities of a fast one
// (0: any number)
static constexpr int lane_waves(int n)
{
    return (n >= JK_FOUR && n < JK_TWO) || n >= JK_TWO + 3 ? 4 : 2;
}
static constexpr int lane_densities(int n)
{
    return n >= JK_TWO ? 2 : n >= JK_FAST && n != JK_FOUR ? 1 : 0;
}
struct ClassInfo {
    bool lane;
    // two wavefronts per work item: FP32 and FP64 queues, FP64 only (the same for
    // teams), one density in FP64: J and K, J, K (JK_FAST + 0, 1, 2); four
    // wavefronts (JK_FOUR on): FP64 only, J and K, K; two densities in FP64 (JK_TWO
    // on): as JK_FAST, and J and K, K with four wavefronts; NULL where the class has
    // none
    const void *fn[JK_KERNELS];
    int threads[JK_KERNELS];
    size_t lds_static[JK_KERNELS];
    int nfij;                   // rows of the K rows
    double cost;                // rough work of one primitive quartet
    // workgroups per CU without dynamic LDS, per device (0: not yet asked);
    // a property of the compiled kernel
    std::atomic<int> *occ[JK_KERNELS];
};

template <int LI, int LJ, int LK, int LL>
static const ClassInfo *class_info()
{
    static std::atomic<int> occ[JK_KERNELS][JK_MAX_DEVICES];
    using T = ClassTraits<LI, LJ, LK, LL>;
    static const ClassInfo info = [] {
        ClassInfo c;
        c.lane = T::LANE;
        c.nfij = ncart(LI) + ncart(LJ);
        c.cost = T::N * (3. * T::NF + 9. * T::GS) + 200.;
        for (int n = 0; n < JK_KERNELS; ++n) { c.occ[n] = occ[n]; c.fn[n] = nullptr; }
        if constexpr (T::LANE) {
            constexpr bool FAST_J = LaneFast<LI, LJ, LK, LL, true>::ON;
            c.fn[0] = (const void *)jk_lane_kernel<LI, LJ, LK, LL, 0, 2>;
            c.fn[1] = (const void *)jk_lane_kernel<LI, LJ, LK, LL, 1, 2>;
            if constexpr (FAST_J) {
                c.fn[2] = (const void *)jk_lane_fast_kernel<LI, LJ, LK, LL, true, true, 2, 1>;
                c.fn[3] = (const void *)jk_lane_fast_kernel<LI, LJ, LK, LL, true, false, 2, 1>;
                c.fn[8] = (const void *)jk_lane_fast_kernel<LI, LJ, LK, LL, true, true, 2, 2>;
                c.fn[9] = (const void *)jk_lane_fast_kernel<LI, LJ, LK, LL, true, false, 2, 2>;
            }
            c.fn[4] = (const void *)jk_lane_fast_kernel<LI, LJ, LK, LL, false, true, 2, 1>;
            c.fn[10] = (const void *)jk_lane_fast_kernel<LI, LJ, LK, LL, false, true, 2, 2>;
            if constexpr (FourWaves<LI, LJ, LK, LL>::ON) {
                c.fn[5] = (const void *)jk_lane_kernel<LI, LJ, LK, LL, 1, 4>;
                if constexpr (FAST_J) {
                    c.fn[6] = (const void *)jk_lane_fast_kernel<LI, LJ, LK, LL, true, true, 4, 1>;
                    c.fn[11] = (const void *)jk_lane_fast_kernel<LI, LJ, LK, LL, true, true, 4, 2>;
                }
                c.fn[7] = (const void *)jk_lane_fast_kernel<LI, LJ, LK, LL, false, true, 4, 1>;
                c.fn[12] = (const void *)jk_lane_fast_kernel<LI, LJ, LK, LL, false, true, 4, 2>;
            }
            for (int n = 0; n < JK_KERNELS; ++n) {
                const int nw = lane_waves(n), nd = lane_densities(n);
                c.threads[n] = nw * WAVE;
                c.lds_static[n] = sizeof(uint32_t) * nw * 2 * 2 * WAVE +
                                  sizeof(double) * MomentRows<T::N>::SIZE +
                                  2 * nd * sizeof(double) * ncart(LI) * ncart(LJ) +
                                  (nd ? 32 : 0);
            }
        } else {
            using S = TeamShape<LI, LJ, LK, LL>;
            c.fn[0] = c.fn[1] = (const void *)jk_team_kernel<LI, LJ, LK, LL>;
            // queue, wave counts, stop flag, team buffers
            const size_t lds = sizeof(uint32_t) * 2 * S::TB + sizeof(int) * (S::TB / WAVE + 2) +
                               sizeof(double) * (S::NQ * (S::PER_QB + S::DSZ) +
                                                 S::NFI * S::NFJ) + 256;
            for (int n = 0; n < JK_KERNELS; ++n) { c.lds_static[n] = lds; c.threads[n] = S::TB; }
        }
        return c;
    }();
    return &info;
}
