'''Which kl column windows the screening objects set up (on the CPU).'''
import pytest


def test_j_engine_sets_up_no_windows():
    '''Windows hold K rows; a J-engine builds J only.'''
    from gpu4pyscf_amd.gto.mole import M
    from gpu4pyscf_amd.scf import j_engine
    opt = j_engine._VHFOpt(M(atom='H 0 0 0; H 0 0 1', basis='sto-3g'))
    assert opt.kl_window_ao == opt.kl_window_ao_team == 0


def _window_sets(policy):
    import torch
    from gpu4pyscf_amd.gto.mole import M
    from gpu4pyscf_amd.gto.sorted_gto import SortedGTO
    from gpu4pyscf_amd.scf import jk
    from oracle import oracle as O
    from tests.molecules import ATOM6
    mol = M(atom=ATOM6, basis='def2-tzvp', unit='B')
    opt = jk._VHFOpt(mol)
    opt.kl_window_ao, opt.kl_window_ao_team, opt.kl_win_policy = 10, 6, policy
    opt.sorted_mol = sm = SortedGTO(mol, diffuse_cutoff=0.3)
    cache = {k: (v[0], v[1], v[1]) for k, v in O.build_pairs(sm).items()}
    dev = {k: torch.as_tensor(v[0].astype('int64')) for k, v in cache.items()}
    return opt, sm, cache, opt._kl_windows(cache, dev, dev, dev)


@pytest.mark.parametrize('policy', [0, 1])
def test_windows_only_for_kets_of_per_lane_classes(policy):
    '''Kets that only team classes have get the windows of the team kernels, under
    the policy that uses them; the others both sets.'''
    from gpu4pyscf_amd.scf import jk
    opt, sm, cache, out = _window_sets(policy)
    ls = sm.uniq_l_ctr[:, 0]
    seen = set()
    for (k, l), (p, _, _) in cache.items():
        lane = jk.has_lane_class(int(ls[k]), int(ls[l]))
        assert lane == ((ls[k], ls[l]) not in ((2, 2), (3, 1), (3, 2), (3, 3)))
        for n, W in enumerate((10, 6)):
            ref = jk.kl_window_table(p, sm.group_offsets, sm.ao_loc, sm.nbas, k, l, W)
            if not (lane or (n == 1 and policy == 1)):
                ref = None
            got = out.get((k, l), [None, None])[n]
            assert (got is None) == (ref is None)
            if ref is not None:
                seen.add((n, lane))
                assert (got[3].numpy() == ref[1]).all() and got[4] == ref[2]
                assert (got[0].numpy() == p[ref[0]]).all()
    assert seen == {(0, True), (1, True)} | ({(1, False)} if policy == 1 else set())


def test_launches_of_other_kets_use_no_windows():
    '''The plan of a class whose ket has no per-lane class is the same with kl
    windows and without.'''
    from gpu4pyscf_amd.lib import clib
    from gpu4pyscf_amd.scf import jk
    from tests.test_launch_plan import _args, _plan, _task
    for li in range(4):
        for lj in range(li + 1):
            for lk in range(li + 1):
                for ll in range(lk + 1):
                    if jk.has_lane_class(lk, ll):
                        continue
                    plans = []
                    for n_win in (0, 5):
                        tasks = (clib.JKTask * 1)()
                        _task(tasks[0], (li, lj, lk, ll), 3000, 5000, n_win=n_win)
                        plans.append([[(x.launch, x.threads, x.block0, x.blocks)
                                       for x in _plan(_args(n_dm, vj, vk, fp32), tasks)]
                                      for n_dm in (1, 2) for vj, vk in ((1, 1), (1, 0), (0, 1))
                                      for fp32 in (False, True)])
                    assert plans[0] == plans[1]


def test_window_defaults_by_name():
    from gpu4pyscf_amd.gto.mole import M
    from gpu4pyscf_amd.scf import jk
    opt = jk._VHFOpt(M(atom='H 0 0 0; H 0 0 1', basis='sto-3g'))
    assert opt.kl_window_ao == jk.KL_WINDOW_AO
    assert opt.kl_window_ao_team == jk.KL_WINDOW_AO_TEAM


def test_kernel_names_of_fp64_builds():
    from gpu4pyscf_amd.scf import jk
    for ls, name in (((1, 0, 1, 0), 'jk_lane_fast_kernel'), ((2, 1, 1, 1), 'jk_lane_fast_kernel'),
                     ((3, 1, 2, 0), 'jk_lane_kernel'), ((3, 0, 2, 1), 'jk_team_kernel'),
                     ((4, 0, 0, 0), 'jk_generic_kernel')):
        args = ', '.join(map(str, ls))
        assert jk.class_kernel_name(ls, 1) == jk.class_kernel_name(ls, 2) == f'{name}<{args}>'
        assert jk.class_kernel_name(ls) == f"{name.replace('fast_', '')}<{args}>"
        assert jk.class_kernel_name(ls, 3) == jk.class_kernel_name(ls)
