'''Batched launches of builds that fill the GPU (cut by workgroups per CU and by
LDS) against one launch per task, and tasks given in two runs of their ij pairs,
as the planner cuts those above the grid limit.  The quartets are the same and
the results differ in the order of the additions only: up to nao^2 terms per
element, so nao^2 x 2.2e-16 of the largest element bounds the difference.'''
import ctypes

import numpy as np
import pytest

from tests.conftest import has_gpu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module', autouse=True)
def _need_gpu():
    if not has_gpu():
        pytest.skip('no HIP device')


def _opt(shape, basis, n_dm, windows=None):
    import torch
    from gpu4pyscf_amd.gto import geometry as G
    from gpu4pyscf_amd.gto.mole import M
    from gpu4pyscf_amd.scf import jk
    print(f'[{shape} water, {basis}, n_dm={n_dm}, windows={windows}]', flush=True)
    mol = M(atom=G.to_string(G.water_cluster(shape, 3., seed=4)), basis=basis)
    opt = jk._VHFOpt(mol)
    if windows:
        opt.kl_window_ao, opt.kl_window_ao_team = windows
    opt.build()
    dm = np.random.default_rng(3).standard_normal((n_dm, mol.nao, mol.nao))
    dm = torch.as_tensor(dm + dm.transpose(0, 2, 1), device='cuda')
    return opt, opt.apply_coeff_C_mat_CT(dm)


def _same(got, ref):
    for x, y in zip(got, ref):
        assert float((x - y).abs().max()) <= x.shape[-1]**2 * 2.2e-16 * float(y.abs().max())


@pytest.mark.parametrize('n_dm', [1, 2])
def test_full_launches_match_one_launch_per_task(n_dm):
    opt, dms = _opt((2, 2, 2), 'def2-tzvp', n_dm)
    kw = dict(count_quartets=True, hash_quartets=True)
    got = opt.get_jk(dms, 1, **kw)
    counts, hashes = opt.last_task_counts, opt.last_task_hashes
    ref = opt.get_jk(dms, 1, time_classes=True, **kw)
    assert counts == opt.last_task_counts and hashes == opt.last_task_hashes
    _same(got, ref)


@pytest.mark.parametrize('shape,basis,n_dm,windows,fp32_tol', [
    ((2, 2, 1), 'def2-tzvp', 1, (96, 48), None), ((2, 2, 1), 'def2-tzvp', 2, None, None),
    ((2, 2, 1), 'def2-tzvp', 1, (96, 48), 1e-4),
    ((2, 1, 1), ('def2-svp', [[4, [.9, 1.]]]), 1, None, None)])
def test_tasks_in_two_runs_of_their_ij_pairs(shape, basis, n_dm, windows, fp32_tol):
    from gpu4pyscf_amd.lib import clib
    opt, dms = _opt(shape, basis, n_dm, windows)
    ref = opt.get_jk(dms, 1, fp32_tol=fp32_tol, count_quartets=True)
    total = opt.last_quartets
    tasks = opt.tasks()
    arr, n = (clib.JKTask * (2 * len(tasks)))(), 0
    for t in range(len(tasks)):
        whole = opt._dev['task_array'][t]
        first = whole.npairs_ij // 2
        for p0, np_ in ((0, first), (first, whole.npairs_ij - first)):
            k = arr[n]
            ctypes.memmove(ctypes.byref(k), ctypes.byref(whole), ctypes.sizeof(k))
            k.npairs_ij = np_
            k.pairs_ij = whole.pairs_ij + 4 * p0
            k.q_ij = whole.q_ij + 4 * p0
            k.pdata_ij = whole.pdata_ij + 48 * whole.iprim * whole.jprim * p0
            n += 1
    opt._dev['task_array'] = arr
    opt.tasks = lambda: list(range(n))
    got = opt.get_jk(dms, 1, fp32_tol=fp32_tol, count_quartets=True)
    assert opt.last_quartets == total
    _same(got, ref)
