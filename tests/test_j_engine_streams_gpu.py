'''Which J-engine calls put their Hermite tasks on side streams, and that the
result does not depend on it: the same sums in another order, up to 1e4 terms
per element.'''
import numpy as np
import pytest

from tests.conftest import has_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('n,basis,n_dm,forks', [(0, 'sto-3g', 1, 0), (1, 'sto-3g', 2, 0),
                                                (2, 'sto-3g', 2, 2), (1, 'def2-svp', 2, 2)])
def test_small_calls_stay_on_the_callers_stream(n, basis, n_dm, forks):
    if not has_gpu():
        pytest.skip('no HIP device')
    import torch
    from gpu4pyscf_amd.gto import geometry as G
    from gpu4pyscf_amd.gto.mole import M
    from gpu4pyscf_amd.scf import j_engine
    atoms = 'H 0 0 0; H 0 0 .74' if n == 0 else G.to_string(G.water_cluster((n, 1, 1), 3., seed=3))
    print(f'[{n} water, {basis}, n_dm={n_dm}]', flush=True)
    mol = M(atom=atoms, basis=basis)
    opt = j_engine._VHFOpt(mol).build()
    calls, fork = [], opt.fork_streams

    def counted(device):
        calls.append(device)
        return fork(device)
    opt.fork_streams = counted
    dm = np.random.default_rng(2).standard_normal((n_dm, mol.nao, mol.nao))
    dm = torch.as_tensor(dm + dm.transpose(0, 2, 1), device='cuda')
    got = j_engine.get_j(mol, dm, vhfopt=opt)
    # (the Rys build forks once more)
    assert len(calls) - bool(opt.tasks()) == forks
    opt.nstreams = 1
    ref = j_engine.get_j(mol, dm, vhfopt=opt)
    assert float((got - ref).abs().max()) <= 1e4 * 2.2e-16 * float(ref.abs().max())
