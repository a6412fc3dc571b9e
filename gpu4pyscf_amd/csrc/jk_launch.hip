// Launch planning: the tasks of a build grouped by angular class into batched
// launches (TaskBatch), spread over the caller's streams.
#include <algorithm>
#include <climits>
#include <map>
#include <mutex>
#include <vector>
#include "jk_launch.h"

// class information, one function per part of the class list (jk_classes.hip)
const ClassInfo *jk_class_info_part0(int key);
const ClassInfo *jk_class_info_part1(int key);
const ClassInfo *jk_class_info_part2(int key);
const ClassInfo *jk_class_info_part3(int key);
const ClassInfo *jk_class_info_part4(int key);
const ClassInfo *jk_class_info_part5(int key);
const ClassInfo *jk_class_info_part6(int key);
const ClassInfo *jk_class_info_part7(int key);

#define JK_TEMPLATED_LMAX 3
// LDS bytes a workgroup may use (static + dynamic): the device limit, capped
// at 64 KB.  gfx950 reports 160 KB per workgroup, but every launch of this
// library stays within the 64 KB that has been validated on the hardware.
#define JK_LDS_CAP (64 * 1024)
// work items per launch that the kl chunks of the per-lane gradient aim at
#define IP1_ITEMS 4096
// kl pairs from which a work item has enough survivors for four wavefronts
// (16 waters, J only: 50 -> 52 ms with four; 8 waters def2-SVP: 2.07 -> 2.46)
#define FOUR_MIN_KL 1024
// densities that the descriptor of a work item can name (TaskDesc.ls_swap)
#define FAST_DM_MAX 32767
// LDS of a gfx950 CU is handed out in units of this many bytes
#define JK_LDS_UNIT 1280

static const ClassInfo *class_info_of(int key)
{
    const ClassInfo *(*const parts[])(int) = {jk_class_info_part0, jk_class_info_part1,
                                              jk_class_info_part2, jk_class_info_part3,
                                              jk_class_info_part4, jk_class_info_part5,
                                              jk_class_info_part6, jk_class_info_part7};
    for (auto f : parts)
        if (const ClassInfo *c = f(key)) return c;
    return nullptr;
}

struct DeviceLimits { int dev; size_t lds_block, lds_cu; int cus; };

static DeviceLimits device_limits()
{
    static std::mutex mu;
    static DeviceLimits known[JK_MAX_DEVICES];
    DeviceLimits l = {-1, JK_LDS_CAP, 160 * 1024, 256};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= JK_MAX_DEVICES) return l;
    std::lock_guard<std::mutex> lock(mu);
    if (known[dev].cus == 0) {
        int v = 0;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) ==
                hipSuccess && v > 0 && v < JK_LDS_CAP)
            l.lds_block = v;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) ==
                hipSuccess && v > 0)
            l.lds_cu = v;
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
            v > 0)
            l.cus = v;
        l.dev = dev;
        known[dev] = l;
    }
    return known[dev];
}

// Workgroups per CU of a class kernel with `bytes` of dynamic LDS: by its
// registers (asked once per kernel and device) and by the LDS of a CU.
static int blocks_per_cu(const ClassInfo &c, int f, size_t bytes, const DeviceLimits &lim)
{
    int nb = lim.dev >= 0 ? c.occ[f][lim.dev].load(std::memory_order_relaxed) : 0;
    if (nb == 0) {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, c.fn[f], c.threads[f], 0) !=
                hipSuccess || nb < 1)
            nb = 1;
        if (lim.dev >= 0) c.occ[f][lim.dev].store(nb, std::memory_order_relaxed);
    }
    const size_t lds = (c.lds_static[f] + bytes + JK_LDS_UNIT - 1) / JK_LDS_UNIT * JK_LDS_UNIT;
    const int by_lds = (int)(lim.lds_cu / lds);
    return std::max(1, std::min(nb, by_lds));
}

// One task, or a run of its ij pairs, in a launch.
struct Item {
    TaskDesc d;
    long blocks;        // the same number for every ij pair
    size_t lds;
    int per_cu;         // workgroups per CU with this LDS
    double cost;        // rough work of the task
};

// LDS K rows of a per-lane task.  Candidates: the rows over the whole k and
// l groups and, when the task has kl column windows, over one window, each
// with and without the density rows.  Ranked by the rows kept in LDS (all
// four K blocks, then K_il/K_jl only, then none), then by the workgroups a
// CU can hold with that LDS, then whole groups before windows, then with
// density rows before without.  kl_win_policy 1 takes the windows whenever
// their rows fit.
static bool plan_lane_rows(const JKBuildArgs &a, const JKTask &k, const ClassInfo &c, int f,
                           const DeviceLimits &lim, Item &it)
{
    // whole kl lists per work item unless that leaves the GPU idle
    int nchunks = (LANE_ITEMS + k.npairs_ij - 1) / k.npairs_ij;
    const int maxchunks = (k.npairs_kl + LANE_MIN_CHUNK - 1) / LANE_MIN_CHUNK;
    nchunks = std::max(1, std::min(nchunks, maxchunks));
    it.d.kl_chunk = (k.npairs_kl + nchunks - 1) / nchunks;
    nchunks = (k.npairs_kl + it.d.kl_chunk - 1) / it.d.kl_chunk;
    it.blocks = (long)k.npairs_ij * nchunks;
    it.d.use_lds = 0;
    it.lds = 0;
    // the fast kernels' copy of the ij primitives
    const int nd = lane_densities(f);
    const bool fast = nd > 0;
    const size_t pij = fast ? (size_t)k.iprim * k.jprim * PIJ_LDS * sizeof(double) : 0;
    // bra blocks of 9 AOs and more on the narrower windows: rows over the wider
    // ones leave one workgroup per CU, or do not fit (48 waters def2-TZVP, one
    // stream, ms, 256 -> 128 AOs: (dp|ps) 34.4 -> 25.6, (fp|ps) 30.9 -> 19.7,
    // (fs|ds) 23.0 -> 17.0, (fp|ss) 17.4 -> 9.1, (dp|ds) 14.8 -> 10.9; 4 to 7 AOs:
    // (ps|ps) 55.9 -> 62.4, (ds|ps) 35.1 -> 41.1, (ds|pp) 31.3 -> 36.2)
    const JKWindows &w = k.kl_win[fast && c.nfij * nd >= 9 && k.kl_win[1].win ? 1 : 0];
    const long blocks_w = w.win ? (long)k.npairs_ij * w.n_win : 0;
    const bool have_win = w.win && LANE_KROWS >= 2;
    long best_key = -1;
    for (int win = 0; win < (have_win ? 2 : 1); ++win) {
        const int kn = win ? w.width : k.k_nao, ln = win ? 0 : k.l_nao;
        for (int dr = (LANE_DROWS || fast ? 1 : 0); dr >= (fast ? 1 : 0); --dr) {
            size_t bytes = 0;
            int mode = 0;
            if (fast && !a.vk) {
                bytes = pij;
                if (c.lds_static[f] + bytes > lim.lds_block) continue;
            } else if (a.vk && (fast || a.n_dm == 1) && kn >= 0 && ln >= 0 && kn + ln > 0) {
                const size_t both = (size_t)c.nfij * (kn + ln) * sizeof(double) * (fast ? nd : 1);
                const size_t lonly = (size_t)c.nfij * ln * sizeof(double);
                if (LANE_KROWS >= 2 && dr && 2 * both + pij + c.lds_static[f] <= lim.lds_block) {
                    mode = 2 | KR_DROWS; bytes = 2 * both + pij;
                } else if (LANE_KROWS >= 2 && !dr && both + c.lds_static[f] <= lim.lds_block) {
                    mode = 2; bytes = both;
                } else if (!win && LANE_KROWS >= 1 && ln > 0 &&
                           lonly + c.lds_static[f] <= lim.lds_block) {
                    mode = 1; bytes = lonly;
                }
            }
            if (win && (mode & KR_MODE_MASK) != 2) continue;
            if (fast && a.vk && !(mode & KR_DROWS)) continue;
            const int nb = blocks_per_cu(c, f, bytes, lim);
            long key = ((long)(mode & KR_MODE_MASK) << 24) | ((long)nb << 8) |
                       ((win ? 0 : 1) << 1) | (dr ? 1 : 0);
            if (a.kl_win_policy == 1 && win) key |= 1L << 30;
            if (key > best_key) {
                best_key = key;
                it.d.use_lds = mode | (win ? KR_WIN : 0);
                it.lds = bytes;
                it.per_cu = nb;
            }
        }
    }
    if (it.d.use_lds & KR_WIN) {
        it.d.pairs_kl = w.pairs; it.d.q_kl = w.q; it.d.pdata_kl = w.pdata; it.d.win = w.win;
        it.blocks = blocks_w;
    }
    return best_key >= 0;
}

// A build in FP64 runs on the kernels compiled for one or two densities
// (JK_FAST, JK_TWO: all rows and the ij primitives in LDS) when their LDS fits;
// returns the kernel, an index of ClassInfo.fn.  n_dm: densities still to do.
static int plan_lane(const JKBuildArgs &a, const JKTask &k, const ClassInfo &c, int pm, int n_dm,
                     const DeviceLimits &lim, Item &it)
{
    const int what = a.vk ? (a.vj ? 0 : 2) : 1;
    // Several densities: only where the last one of an odd number fits too, and
    // not in several launches of a task that leaves CUs idle, which take the
    // time of one each (1 water def2-TZVP, three densities: 7.6 -> 10.6 ms).
    // Two densities, ms, any-number kernel -> this: 8 waters def2-SVP 6.6 -> 3.4,
    // 8 and 12 waters def2-TZVP 53.6 -> 36.1 and 143 -> 75; 12 waters in two
    // launches of one density 92.
    // J only of more than two densities: s and p classes stay on the any-number
    // kernel, whose J costs less than evaluating their integrals again for each two
    // (eight densities, ms, in pairs -> together: 64 waters STO-3G 117 -> 95 on one
    // stream, all s and p; 32 waters def2-SVP (ps|ss) 36.2 -> 30.1, (ss|ss) 21.0 ->
    // 17.1, but (dp|ps) 8.7 -> 14.6, (dp|ds) 2.3 -> 5.6, (dp|ss) 3.9 -> 6.0).
    const bool together = !a.vk && a.n_dm > 2 && k.li <= 1;
    Item one = it;
    const bool fast = pm == 1 && !together &&
                      (a.n_dm == 1 || (a.n_dm <= FAST_DM_MAX && c.fn[JK_FAST + what] &&
                                       plan_lane_rows(a, k, c, JK_FAST + what, lim, one) &&
                                       (a.n_dm == 2 || one.blocks > lim.cus)));
    const bool two = fast && n_dm >= 2;
    const bool four = fast && a.vk && k.npairs_kl >= FOUR_MIN_KL;
    // in order of preference
    const int tries[] = {two && four ? JK_TWO + (a.vj ? 3 : 4) : -1, two ? JK_TWO + what : -1,
                         four ? JK_FOUR + (a.vj ? 1 : 2) : -1, fast ? JK_FAST + what : -1,
                         four && a.n_dm == 1 ? JK_FOUR : -1, pm};
    for (int f : tries)
        if (f >= 0 && c.fn[f] && plan_lane_rows(a, k, c, f, lim, it)) return f;
    return pm;
}

static void plan_team(const JKBuildArgs &a, const JKTask &k, const ClassInfo &c,
                      const DeviceLimits &lim, Item &it)
{
    it.d.kl_chunk = TEAM_KL_CHUNK;
    it.blocks = (long)k.npairs_ij * ((k.npairs_kl + TEAM_KL_CHUNK - 1) / TEAM_KL_CHUNK);
    it.d.use_lds = 0;
    it.lds = 0;
    const JKWindows &w = k.kl_win[1];
    if (w.win && a.vk && a.n_dm == 1 && (TEAM_KWIN || a.kl_win_policy == 1)) {
        // K rows over one kl column window per work item, when that leaves
        // enough work items to fill the GPU
        const size_t bytes = sizeof(double) * c.nfij * (size_t)w.width;
        const long blocks_w = (long)k.npairs_ij * w.n_win;
        if (bytes + c.lds_static[1] <= lim.lds_block &&
            (a.kl_win_policy == 1 || blocks_w >= TEAM_KWIN_MIN_ITEMS)) {
            it.d.pairs_kl = w.pairs; it.d.q_kl = w.q; it.d.pdata_kl = w.pdata; it.d.win = w.win;
            it.d.use_lds = 2 | KR_WIN;
            it.blocks = blocks_w;
            it.lds = bytes;
        }
    }
    if (!(it.d.use_lds & KR_WIN) && TEAM_KROWS >= 1 && a.vk && a.n_dm == 1 && k.l_nao > 0) {
        const size_t bytes = sizeof(double) * c.nfij * (size_t)k.l_nao;
        if (bytes + c.lds_static[1] <= lim.lds_block) { it.d.use_lds = 1; it.lds = bytes; }
    }
    it.per_cu = blocks_per_cu(c, 1, it.lds, lim);
}

// A kernel of this library and how it is launched.
struct Kernel {
    const void *fn;
    int threads;
    // 0 the whole operator; 1 and 2 its attenuated and its full-range part, for
    // the kernels that take one at a time (runtime l; per-lane ones with J)
    int part;
};

struct Launch {
    Kernel k;
    TaskBatch b;
    long blocks;
    size_t lds;
    double cost;
};

// Workgroups of one launch: a grid holds fewer than 2^32 threads (the dispatch
// packet counts them in 32 bits), and the kernels count workgroups in an int.
static long max_blocks(int threads)
{
    return std::min((long)INT_MAX, (long)UINT32_MAX / threads);
}

// Appends an item; one above the limit of a launch in runs of its ij pairs.
// false when the workgroups of one ij pair exceed it.
static bool add_item(std::vector<Item> &items, const Item &it, int threads)
{
    const int npairs = it.d.npairs_ij;
    const long most = max_blocks(threads), per_pair = it.blocks / npairs;
    if (per_pair > most) return false;
    const int step = (int)std::min((long)npairs, most / per_pair);
    const int nij = (it.d.prims_ij & 0xffff) * (it.d.prims_ij >> 16);
    for (long p0 = 0; p0 < npairs; p0 += step) {
        Item part = it;
        TaskDesc &d = part.d;
        d.npairs_ij = (int)std::min((long)step, npairs - p0);
        d.pairs_ij += p0;
        d.q_ij += p0;
        d.pdata_ij += p0 * nij * PREC;
        part.blocks = per_pair * d.npairs_ij;
        part.cost = it.cost * d.npairs_ij / npairs;
        items.push_back(part);
    }
    return true;
}

// Cuts the items of one kernel into launches.  Items with the same LDS need go
// together; others only join when the whole class leaves CUs idle anyway,
// so that no item is held to the workgroups per CU of a wider one.
static void make_launches(std::vector<Item> &items, const Kernel &kernel, int cus,
                          std::vector<Launch> &out)
{
    long total = 0;
    int per_cu = INT_MAX;
    for (const Item &it : items) {
        total += it.blocks;
        per_cu = std::min(per_cu, it.per_cu);
    }
    const bool merge = total <= (long)cus * per_cu;
    // the longest work items first: they start first, the short ones fill
    // the tail
    std::stable_sort(items.begin(), items.end(), [&](const Item &x, const Item &y) {
        if (!merge && x.per_cu != y.per_cu) return x.per_cu < y.per_cu;
        return x.cost / x.blocks > y.cost / y.blocks;
    });
    int last_cu = 0;
    for (const Item &it : items) {
        if (last_cu == 0 || out.back().b.n == JK_BATCH || (!merge && it.per_cu != last_cu) ||
            out.back().blocks + it.blocks > max_blocks(kernel.threads)) {
            out.push_back(Launch());
            Launch &l = out.back();
            l.k = kernel;
            l.b.n = l.b.pad = 0;
            std::fill(l.b.block0, l.b.block0 + JK_BATCH + 1, INT_MAX);
            l.blocks = 0;
            l.lds = 0;
            l.cost = 0.;
        }
        last_cu = it.per_cu;
        Launch &l = out.back();
        l.b.t[l.b.n] = it.d;
        l.b.block0[l.b.n++] = (int)l.blocks;
        l.blocks += it.blocks;
        l.lds = std::max(l.lds, it.lds);
        l.cost += it.cost;
    }
}

static hipError_t plan_tasks(const JKBuildArgs &a, const JKTask *tasks, int ntasks,
                             const JKRun &run, std::vector<Launch> &launches)
{
    const DeviceLimits lim = device_limits();
    const int pm = a.fp32_cut > -1e29f ? 0 : 1;
    // items by kernel, the classes of the last tasks (f shells) first; the
    // key of the runtime-l kernel is -1
    struct Group { Kernel k; std::vector<Item> items; };
    std::map<int, Group> by_kernel;
    std::vector<int> order;
    auto add = [&](int key, const Kernel &kern, const Item &it) {
        Group &g = by_kernel[3 * key + kern.part];
        if (g.items.empty()) {
            order.push_back(3 * key + kern.part);
            g.k = kern;
        }
        return add_item(g.items, it, kern.threads);
    };
    for (int t = ntasks - 1; t >= 0; --t) {
        const JKTask &k = tasks[t];
        if (k.npairs_ij <= 0 || k.npairs_kl <= 0) continue;
        Item it;
        TaskDesc &d = it.d;
        d.pairs_ij = k.pairs_ij; d.pairs_kl = k.pairs_kl;
        d.q_ij = k.q_ij; d.q_kl = k.q_kl;
        d.pdata_ij = k.pdata_ij; d.pdata_kl = k.pdata_kl;
        d.win = nullptr;
        d.npairs_ij = k.npairs_ij; d.npairs_kl = k.npairs_kl;
        d.prims_ij = k.iprim | (uint32_t)k.jprim << 16;
        d.prims_kl = k.kprim | (uint32_t)k.lprim << 16;
        d.k_ao0 = k.k_ao0; d.k_nao = k.k_nao; d.l_ao0 = k.l_ao0; d.l_nao = k.l_nao;
        d.counter = t;
        d.ls_swap = k.li | k.lj << 4 | k.lk << 8 | k.ll << 12 | (k.swap_ijkl != 0) << 16;
        d.use_lds = 0;
        const double quartets = (double)k.npairs_ij * k.npairs_kl * k.iprim * k.jprim * k.kprim *
                                k.lprim;
        int key = k.li * 125 + k.lj * 25 + k.lk * 5 + k.ll;
        const bool small = k.li <= JK_TEMPLATED_LMAX && k.lj <= JK_TEMPLATED_LMAX &&
                           k.lk <= JK_TEMPLATED_LMAX && k.ll <= JK_TEMPLATED_LMAX;
        const void *ip1 = run.mode != GEN_JK && small ? jk_ip1_lane_kernel_of(key) : nullptr;
        Kernel kern;
        if (ip1) {
            kern = {ip1, WAVE, 0};
            const int nchunks = std::min((IP1_ITEMS + k.npairs_ij - 1) / k.npairs_ij,
                                         (k.npairs_kl + WAVE - 1) / WAVE);
            d.kl_chunk = (k.npairs_kl + nchunks - 1) / nchunks;
            it.blocks = (long)k.npairs_ij * ((k.npairs_kl + d.kl_chunk - 1) / d.kl_chunk);
            it.lds = 0;
            it.per_cu = 4;
            it.cost = quartets * ncart(k.li) * ncart(k.lj) * ncart(k.lk) * ncart(k.ll);
        } else if (run.mode != GEN_JK || !small) {
            key = -1;
            kern = {jk_generic_kernel_of(run.mode), GEN_TB, 0};
            if (!jk_generic_plan(k, run.mode, d, it.blocks, it.lds)) return hipErrorNotSupported;
            it.per_cu = (int)(lim.lds_cu / (it.lds + 4096));
            it.cost = quartets * ncart(k.li) * ncart(k.lj) * ncart(k.lk) * ncart(k.ll);
            if (run.mode == GEN_JK && a.full != 0.) kern.part = 1;
        } else {
            const ClassInfo *c = class_info_of(key);
            if (!c) return hipErrorNotSupported;
            it.cost = quartets * c->cost * (a.full != 0. ? 2 : 1);
            if (c->lane) {
                // the fast kernels in as many launches as the densities take
                for (int dm0 = 0; dm0 < a.n_dm;) {
                    Item part = it;
                    const int f = plan_lane(a, k, *c, pm, a.n_dm - dm0, lim, part);
                    const int nd = lane_densities(f);
                    if (nd) part.d.ls_swap |= (uint32_t)dm0 << 17;
                    const bool split = a.full != 0. && !(nd && !a.vj);
                    for (int p = split ? 1 : 0; p <= (split ? 2 : 0); ++p)
                        if (!add(key * JK_KERNELS + f, {c->fn[f], c->threads[f], p}, part))
                            return hipErrorInvalidConfiguration;
                    dm0 += nd ? nd : a.n_dm;
                }
                continue;
            }
            plan_team(a, k, *c, lim, it);
            kern = {c->fn[pm], c->threads[pm], 0};
            key = key * JK_KERNELS + pm;
        }
        if (!add(key, kern, it)) return hipErrorInvalidConfiguration;
        if (kern.part == 1) {
            kern.part = 2;
            if (!add(key, kern, it)) return hipErrorInvalidConfiguration;
        }
    }
    for (int key : order)
        make_launches(by_kernel[key].items, by_kernel[key].k, lim.cus, launches);
    return hipSuccess;
}

hipError_t jk_plan_launches(const JKBuildArgs &a, const JKTask *tasks, int ntasks,
                            const JKRun &run, JKPlanItem *out, int nmax, int &n)
{
    std::vector<Launch> launches;
    const hipError_t err = plan_tasks(a, tasks, ntasks, run, launches);
    if (err != hipSuccess) return err;
    n = 0;
    for (size_t l = 0; l < launches.size(); ++l) {
        const Launch &la = launches[l];
        for (int i = 0; i < la.b.n; ++i, ++n) {
            if (n >= nmax) continue;
            const TaskDesc &d = la.b.t[i];
            const long end = i + 1 < la.b.n ? la.b.block0[i + 1] : la.blocks;
            out[n] = JKPlanItem{(int)l, la.k.threads, la.k.part, d.counter,
                                (int)(d.pairs_ij - tasks[d.counter].pairs_ij), d.npairs_ij,
                                la.b.block0[i], end - la.b.block0[i]};
        }
    }
    return hipSuccess;
}

hipError_t jk_launch_tasks(const JKBuildArgs &a, const JKTask *tasks, int ntasks,
                           void *const *streams, int nstreams, const JKRun &run)
{
    std::vector<Launch> launches;
    const hipError_t planned = plan_tasks(a, tasks, ntasks, run, launches);
    if (planned != hipSuccess) return planned;
    // each launch on the stream with the least work so far, in class order
    // (sorted by the estimate: 54 -> 60 ms on the 8-water two-density build;
    // round-robin: the 16-water range-separated K 144 -> 148 ms)
    std::vector<double> load(nstreams, 0.);
    for (Launch &l : launches) {
        const int s = (int)(std::min_element(load.begin(), load.end()) - load.begin());
        load[s] += l.cost;
        JKBuildArgs p = a;
        if (l.k.part) p.full = 0.;
        if (l.k.part == 2) {
            p.scale = a.scale * a.full;
            p.omega = 0.;
            p.n_quartets = p.n_quartets_fp32 = p.quartet_hash = nullptr;
        }
        void *args[] = {&p, &l.b, (void *)&run.ex};
        const hipError_t err = hipLaunchKernel(l.k.fn, dim3((unsigned)l.blocks),
                                               dim3(l.k.threads), args, l.lds,
                                               (hipStream_t)streams[s]);
        if (err != hipSuccess) return err;
    }
    return hipSuccess;
}
