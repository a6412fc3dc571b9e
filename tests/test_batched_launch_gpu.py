'''Batched class launches (many tasks of one angular class per launch, the
runtime-l kernel's row slices and candidate chunks) against one launch per
task.  The two differ in the order of the additions only: up to 1e4 terms per
element, so 1e4 x 2.2e-16 of the largest element bounds the difference.'''
import ctypes

import numpy as np
import pytest

from tests.conftest import has_gpu

pytestmark = pytest.mark.gpu
TOL = 1e4 * 2.2e-16


@pytest.fixture(scope='module', autouse=True)
def _need_gpu():
    if not has_gpu():
        pytest.skip('no HIP device')


def _mol(n, basis):
    from gpu4pyscf_amd.gto import geometry as G
    from gpu4pyscf_amd.gto.mole import M
    return M(atom=G.to_string(G.water_cluster((n, 1, 1), 3., seed=3)), basis=basis)


G_BASIS = ('def2-svp', [[4, [.9, 1.]]])


@pytest.mark.parametrize('n,basis,n_dm,hermi', [
    (1, 'sto-3g', 1, 1), (1, 'def2-svp', 3, 1), (3, 'def2-svp', 1, 0), (2, 'def2-tzvp', 1, 1),
    (1, 'def2-tzvp', 2, 1), (1, G_BASIS, 2, 1)])
def test_batched_build_matches_one_launch_per_task(n, basis, n_dm, hermi):
    import torch
    from gpu4pyscf_amd.scf import jk
    mol = _mol(n, basis)
    print(f'[{n} water, {basis}, n_dm={n_dm}, hermi={hermi}]', flush=True)
    opt = jk._VHFOpt(mol).build()
    rng = np.random.default_rng(5)
    dm = rng.standard_normal((n_dm, mol.nao, mol.nao))
    if hermi == 1:
        dm = dm + dm.transpose(0, 2, 1)
    dms = opt.apply_coeff_C_mat_CT(torch.as_tensor(dm, device='cuda'))
    got = opt.get_jk(dms, hermi, count_quartets=True, hash_quartets=True)
    counts, hashes = opt.last_task_counts, opt.last_task_hashes
    ref = opt.get_jk(dms, hermi, count_quartets=True, hash_quartets=True, time_classes=True)
    assert counts == opt.last_task_counts and hashes == opt.last_task_hashes
    for x, y in zip(got, ref):
        assert float((x - y).abs().max()) <= TOL * float(y.abs().max())


@pytest.mark.parametrize('basis,n_dm', [('def2-svp', 1), ('def2-svp', 2), ('def2-tzvp', 1),
                                        (G_BASIS, 1)])
def test_gradient_tasks_match_one_launch_per_task(basis, n_dm):
    import torch
    from gpu4pyscf_amd.grad import rhf
    from gpu4pyscf_amd.lib import clib
    mol = _mol(2 if basis == 'def2-svp' else 1, basis)
    print(f'[{basis}, n_dm={n_dm}]', flush=True)
    opt = rhf._VHFOpt(mol).build()
    rng = np.random.default_rng(6)
    dm = rng.standard_normal((n_dm, mol.nao, mol.nao))
    dm = dm + dm.transpose(0, 2, 1)
    de = rhf._jk_energy_per_atom(opt, dm, .8, .6)
    # one jk_energy_ip1 call per task, through a stand-in for the batched entry
    lib, calls = clib.load(), []

    def per_task(args, tasks, ntasks, ejk, copies, stride, jf, kf, streams, nstreams):
        a = args._obj
        for t in range(ntasks):
            for f, _ in clib.JKTask._fields_:
                setattr(a, f, getattr(tasks[t], f))
            st = lib.jk_energy_ip1(ctypes.byref(a), ctypes.c_void_p(ejk), jf, kf, None)
            calls.append(st)
            assert st == 0
        torch.cuda.synchronize()
        return 0

    class Stub:
        def __getattr__(self, name):
            return per_task if name == 'jk_energy_ip1_tasks' else getattr(lib, name)
    loaded, clib._lib = clib._lib, Stub()
    try:
        ref = rhf._jk_energy_per_atom(opt, dm, .8, .6)
    finally:
        clib._lib = loaded
    assert len(calls) == len(opt.tasks())
    assert abs(de - ref).max() <= TOL * abs(ref).max()
