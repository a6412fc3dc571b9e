'''No density at all: the J-engine refuses it as get_jk does, where it has
classes for the Rys build.'''
import pytest

from tests.conftest import has_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('engine', ['jk', 'j_engine'])
def test_no_density_is_refused(engine):
    if not has_gpu():
        pytest.skip('no HIP device')
    import torch
    from gpu4pyscf_amd.gto.mole import M
    from gpu4pyscf_amd.scf import j_engine, jk
    mol = M(atom='O 0 0 0.1174; H -0.757 0 -0.4696; H 0.757 0 -0.4696', basis='def2-svp')
    dm = torch.zeros((0, mol.nao, mol.nao), dtype=torch.float64, device='cuda')
    with pytest.raises(RuntimeError):
        (jk if engine == 'jk' else j_engine).get_j(mol, dm, hermi=1)
