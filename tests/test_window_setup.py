'''Which kl column windows the screening objects set up (on the CPU).'''


def test_j_engine_sets_up_no_windows():
    '''Windows hold K rows; a J-engine builds J only.'''
    from gpu4pyscf_amd.gto.mole import M
    from gpu4pyscf_amd.scf import j_engine
    opt = j_engine._VHFOpt(M(atom='H 0 0 0; H 0 0 1', basis='sto-3g'))
    assert opt.kl_window_ao == opt.kl_window_ao_team == 0
