'''Builds of several densities (kernels of two densities, the odd last one, and
the any-number kernel of small tasks) against builds of one density.  The
densities D, -D and 0 share one screening table, so the quartets are the same
and the results differ in the order of the additions only: up to 1e4 terms per
element, so 1e4 x 2.2e-16 of the largest element bounds the difference.'''
import numpy as np
import pytest

from tests.conftest import has_gpu

pytestmark = pytest.mark.gpu
TOL = 1e4 * 2.2e-16


@pytest.mark.parametrize('shape,basis', [((1, 1, 1), 'def2-svp'), ((3, 1, 1), 'def2-tzvp'),
                                         ((2, 2, 3), 'def2-tzvp')])
@pytest.mark.parametrize('n_dm', [2, 3])
@pytest.mark.parametrize('screen', ['jk', 'j', 'k'])
def test_densities_together_match_one_by_one(shape, basis, n_dm, screen):
    if not has_gpu():
        pytest.skip('no HIP device')
    import torch
    from gpu4pyscf_amd.gto import geometry as G
    from gpu4pyscf_amd.gto.mole import M
    from gpu4pyscf_amd.scf import jk
    print(f'[{shape} water, {basis}, n_dm={n_dm}, screen={screen}]', flush=True)
    mol = M(atom=G.to_string(G.water_cluster(shape, 3., seed=4)), basis=basis)
    opt = jk._VHFOpt(mol).build()
    dm = np.random.default_rng(9).standard_normal((mol.nao, mol.nao))
    dm = opt.apply_coeff_C_mat_CT(torch.as_tensor(dm + dm.T, device='cuda')[None])
    kw = dict(with_j=screen != 'k', with_k=screen != 'j', screen=screen, count_quartets=True,
              hash_quartets=True)
    ref = opt.get_jk(dm, 1, **kw)
    counts, hashes = opt.last_task_counts, opt.last_task_hashes
    sign = torch.tensor([1., -1., 0.][:n_dm], dtype=dm.dtype, device=dm.device)[:, None, None]
    got = opt.get_jk(dm * sign, 1, **kw)
    assert opt.last_task_counts == counts and opt.last_task_hashes == hashes
    for x, y in zip(got, ref):
        if y is not None:
            assert float((x - y * sign).abs().max()) <= TOL * float(y.abs().max())
