'''The launch planner on the CPU (jk_plan_tasks): no launch may hold 2^32 or
more work items (threads), the limit of a HIP grid, and the launches of a build
hold every task's ij pairs once.  Pair counts are synthetic: the lists are never
read.'''
import ctypes

import pytest

LIMIT = 2**32 - 1
ADDR = 1 << 20          # stands for device memory that the planner does not read


def _args(n_dm=1, vj=True, vk=True, fp32=False, omega=0., full=0.):
    from gpu4pyscf_amd.lib import clib
    _, meta = clib.load_rys_table_host()
    a = clib.JKBuildArgs()
    a.abi_version = clib.JK_ABI_VERSION
    for f in ('bas', 'env', 'ao_loc', 'dm_cond', 'dm'):
        setattr(a, f, ADDR)
    a.vj, a.vk = ADDR if vj else None, ADDR if vk else None
    a.nbas, a.nao, a.n_dm = 60000, 40000, n_dm
    a.n_repl = 1
    a.fp32_cut = -10. if fp32 else -1e30
    a.omega, a.full = omega, full
    a.rys.coef = a.rys.coef32 = ADDR
    a.rys.degree, a.rys.boys, a.rys.boys_rows = meta['degree'], meta['boys'], meta['boys_rows']
    a.rys.boys_step = meta['boys_step']
    for n, x in enumerate(meta['xmax']):
        a.rys.xmax[n] = float(x)
    return a


def _task(t, ls, npairs_ij, npairs_kl, nprim=1, n_win=0, nao=4000):
    t.li, t.lj, t.lk, t.ll = ls
    t.iprim = t.jprim = t.kprim = t.lprim = nprim
    t.k_nao = t.l_nao = nao
    t.npairs_ij, t.npairs_kl = npairs_ij, npairs_kl
    for f in ('pairs_ij', 'pairs_kl', 'q_ij', 'q_kl', 'pdata_ij', 'pdata_kl'):
        setattr(t, f, ADDR)
    for n, width in enumerate((300, 200)):
        if n_win:
            w = t.kl_win[n]
            w.pairs = w.q = w.pdata = w.win = ADDR
            w.n_win, w.width = n_win * (n + 1), width


def _plan(args, tasks, gradient=0):
    from gpu4pyscf_amd.lib import clib
    lib = clib.load()
    n = ctypes.c_int()
    st = lib.jk_plan_tasks(ctypes.byref(args), tasks, len(tasks), gradient, None, 0,
                           ctypes.byref(n))
    assert st == 0, lib.jk_last_error()
    out = (clib.JKPlanItem * n.value)()
    assert lib.jk_plan_tasks(ctypes.byref(args), tasks, len(tasks), gradient, out, n.value,
                             ctypes.byref(n)) == 0
    return list(out)


def _check(args, tasks, gradient=0, times=1):
    '''times: launches that hold each ij pair of a task (several densities,
    parts of an operator).'''
    items = _plan(args, tasks, gradient)
    end = {}
    for x in items:
        assert x.blocks > 0 and x.block0 == end.get(x.launch, 0)
        end[x.launch] = x.block0 + x.blocks
        assert end[x.launch] * x.threads <= LIMIT, (end[x.launch], x.threads)
    for t, task in enumerate(tasks):
        runs = [(x.pair0, x.pair0 + x.npairs) for x in items if x.task == t]
        cuts = sorted({0, task.npairs_ij} | {c for r in runs for c in r})
        assert cuts[0] == 0 and cuts[-1] == task.npairs_ij
        for c in cuts[:-1]:
            assert sum(lo <= c < hi for lo, hi in runs) == times, c
    return items


# the classes of one kernel over many group pairs: tasks far below the limit
# whose sum exceeds it
@pytest.mark.parametrize('ls,gradient,npairs,n_win', [
    ((1, 0, 1, 0), 0, 400000, 64),          # per lane, kl windows
    ((3, 0, 2, 1), 0, 60000, 0),            # teams
    ((4, 1, 2, 0), 0, 16000, 0),            # runtime l
    ((2, 2, 2, 1), 1, 20000, 0),            # gradient on the runtime-l kernel
])
def test_batches_stay_below_the_grid_limit(ls, gradient, npairs, n_win):
    from gpu4pyscf_amd.lib import clib
    tasks = (clib.JKTask * 31)()
    for t in tasks:
        _task(t, ls, npairs, npairs, n_win=n_win)
    items = _check(_args(), tasks, gradient)
    assert sum(x.blocks * x.threads for x in items) > LIMIT


# one task above the limit by itself; the last pair counts leave a remainder
@pytest.mark.parametrize('ls,gradient,n_ij,n_kl,n_win', [
    ((1, 0, 0, 0), 0, 900001, 900001, 100), ((3, 0, 2, 1), 0, 400003, 400003, 0),
    ((3, 3, 3, 3), 0, 200000, 300001, 0), ((4, 4, 4, 4), 0, 50000, 70001, 0),
    ((5, 5, 5, 5), 1, 30011, 40000, 0), ((2, 1, 1, 0), 1, 2000003, 2000003, 0)])
def test_large_tasks_are_split_along_their_ij_pairs(ls, gradient, n_ij, n_kl, n_win):
    from gpu4pyscf_amd.lib import clib
    tasks = (clib.JKTask * 2)()
    _task(tasks[0], ls, n_ij, n_kl, n_win=n_win)
    _task(tasks[1], ls, 7, 5, n_win=n_win and 1)
    _check(_args(), tasks, gradient)


@pytest.mark.parametrize('n_dm,vj,vk,fp32,omega,full,times', [
    (2, True, True, False, 0., 0., 1), (3, True, True, False, 0., 0., 2),
    (1, True, True, True, 0., 0., 1), (1, True, True, False, .3, -1., 2),
    (2, False, True, False, .3, -1., 1)])
def test_densities_and_parts_of_large_tasks(n_dm, vj, vk, fp32, omega, full, times):
    from gpu4pyscf_amd.lib import clib
    tasks = (clib.JKTask * 3)()
    for n, t in enumerate(tasks):
        _task(t, (1, 0, 1, 0), 700001 + n, 700001, n_win=90)
    _check(_args(n_dm, vj, vk, fp32, omega, full), tasks, times=times)


def test_plan_of_nothing_and_bad_arguments():
    from gpu4pyscf_amd.lib import clib
    lib = clib.load()
    n = ctypes.c_int(7)
    a = _args()
    tasks = (clib.JKTask * 1)()
    assert lib.jk_plan_tasks(ctypes.byref(a), tasks, 1, 0, None, 0, ctypes.byref(n)) == 0
    assert n.value == 0         # an empty pair list
    assert lib.jk_plan_tasks(ctypes.byref(a), tasks, 1, 0, None, 0, None) == 1
    assert lib.jk_plan_tasks(ctypes.byref(a), tasks, 1, 0, None, 3, ctypes.byref(n)) == 1
    _task(tasks[0], (clib.JK_LMAX + 1, 0, 0, 0), 3, 3)
    assert lib.jk_plan_tasks(ctypes.byref(a), tasks, 1, 0, None, 0, ctypes.byref(n)) == 2


# J of many densities: classes of s and p shells digest all of them beside one
# evaluation of the integrals, the others in pairs
@pytest.mark.parametrize('ls,vk,times', [((0, 0, 0, 0), False, 1), ((1, 1, 1, 0), False, 1),
                                         ((2, 0, 1, 0), False, 3), ((1, 1, 1, 0), True, 3)])
def test_many_densities_evaluate_the_integrals_once_where_that_is_faster(ls, vk, times):
    from gpu4pyscf_amd.lib import clib
    tasks = (clib.JKTask * 1)()
    _task(tasks[0], ls, 20000, 20000, nao=100)
    _check(_args(n_dm=6, vk=vk), tasks, times=times)
    _check(_args(n_dm=2, vk=vk), tasks)
