'''Cases that time the J/K engine through its public entry points.

Each case is one call of a kind that programs on this engine make, with the
molecule, its screening object and the density matrices in hand:

* ``jk``     get_jk: the Fock build of an SCF cycle (one density), of an
             unrestricted SCF (two), or of a response solver (hermi = 0);
* ``mixed``  the same build with FP32 quartets below a bound, the option that
             the SCF driver uses for incremental builds;
* ``rsh_k``  get_k of a range-separated hybrid;
* ``j_md``   get_j of the McMurchie-Davidson J-engine;
* ``grad``   the two-electron part of a nuclear gradient;
* ``scf``    a whole closed-shell SCF from the molecule to the converged
             density, screening setup and one-electron integrals included.

Molecules are the seeded water clusters and alkane chains of
gpu4pyscf_amd.gto.geometry in def2-SVP and def2-TZVP, and def2-TZVP with a g
shell on every atom.
'''
import math

import numpy as np
import torch

from gpu4pyscf_amd.grad import rhf as grad_rhf
from gpu4pyscf_amd.gto import geometry
from gpu4pyscf_amd.gto.mole import M
from gpu4pyscf_amd.scf import j_engine, jk
from gpu4pyscf_amd.scf.hf import RHF

SVP, TZVP, TZVP_G = 'def2-svp', 'def2-tzvp', 'def2-tzvp+g'


def _case(name, kind, system, n, basis, density='delta', n_dm=1, hermi=1, geom=0):
    c = dict(kind=kind, system=system, n=n, basis=basis, density=density, n_dm=n_dm,
             hermi=hermi, geom=geom)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: one molecule, where launches and host work count
        _case('water1_svp_jk', 'jk', 'water', 1, SVP),
        # an ordinary small cluster, one incremental SCF build
        _case('water8_svp_jk', 'jk', 'water', 8, SVP),
        # a medium cluster in the basis of production work
        _case('water32_tzvp_jk', 'jk', 'water', 32, TZVP),
        # the largest: a cluster where every loop is long
        _case('water48_tzvp_jk', 'jk', 'water', 48, TZVP),
        # a chain: sparse pair lists, a density that decays along the molecule
        _case('alkane30_tzvp_jk', 'jk', 'alkane', 30, TZVP, density='full'),
        # an unrestricted SCF builds J and K of two densities at once
        _case('water8_tzvp_uhf', 'jk', 'water', 8, TZVP, density='full', n_dm=2),
        # the mixed-precision incremental build
        _case('water16_tzvp_mixed', 'mixed', 'water', 16, TZVP),
        # exchange of a range-separated hybrid
        _case('water16_tzvp_rsh_k', 'rsh_k', 'water', 16, TZVP, density='full'),
        # Coulomb only, as a pure functional needs it
        _case('water16_tzvp_j_md', 'j_md', 'water', 16, TZVP, density='full'),
        # one step of a geometry optimisation
        _case('water4_svp_grad', 'grad', 'water', 4, SVP, density='full'),
        # a basis with g shells (the runtime-l kernel)
        _case('water1_tzvp_g_jk', 'jk', 'water', 1, TZVP_G, density='full'),
        # a whole SCF of a small cluster
        _case('water8_svp_scf', 'scf', 'water', 8, SVP),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    '''One more case: sizes spread over their logarithm, odd ones among them.'''
    kind = rng.choice(['jk', 'jk', 'jk', 'jk', 'mixed', 'rsh_k', 'j_md', 'grad', 'scf'])
    geom = rng.randrange(1, 1 << 20)
    density = rng.choice(['delta', 'full'])
    if kind in ('grad', 'scf'):
        return _case(None, kind, 'water', rng.randint(1, 4 if kind == 'grad' else 8), SVP, 'full',
                     geom=geom)
    if kind in ('rsh_k', 'j_md', 'mixed'):
        return _case(None, kind, 'water', _log_int(rng, 1, 18), rng.choice([SVP, TZVP]),
                     'delta' if kind == 'mixed' else density, geom=geom)
    which = rng.choice(['one', 'one', 'one', 'alkane', 'several', 'g'])
    if which == 'g':
        return _case(None, kind, 'water', rng.randint(1, 2), TZVP_G, density, geom=geom)
    if which == 'alkane':
        return _case(None, kind, 'alkane', _log_int(rng, 2, 30), rng.choice([SVP, TZVP]),
                     density, geom=geom)
    if which == 'several':
        return _case(None, kind, 'water', _log_int(rng, 1, 10), rng.choice([SVP, TZVP]), 'full',
                     n_dm=rng.choice([1, 2, 3]), hermi=rng.choice([1, 0]), geom=geom)
    return _case(None, kind, 'water', _log_int(rng, 1, 36), rng.choice([SVP, TZVP]), density,
                 geom=geom)


# -- inputs ---------------------------------------------------------------
RSH = dict(omega=.3, lr_factor=.65, sr_factor=.2)   # a range-separated hybrid's exchange
FP32_TOL = 1e-6
DIRECT_SCF_TOL = 1e-13


def _molecule(case, geom):
    if case['system'] == 'alkane':
        atoms = geometry.alkane(case['n'], seed=geom)
    else:
        n = case['n']
        side = max(1, math.ceil(n ** (1. / 3.) - 1e-9))
        shape = (side, side, math.ceil(n / side**2))
        shape = {8: (2, 2, 2), 16: (2, 2, 4), 32: (4, 4, 2), 48: (4, 4, 3)}.get(n, shape)
        # lattice spacing: 3.0 Angstrom up to 32 molecules, 3.1 above
        atoms = geometry.water_cluster(shape, 3. if n <= 32 else 3.1, seed=geom)[:3 * n]
    basis = (TZVP, [[4, [1., 1.]]]) if case['basis'] == TZVP_G else case['basis']
    return M(atom=geometry.to_string(atoms), basis=basis)


def _ao_centres(mol):
    loc = mol.ao_loc
    centre = np.empty((mol.nao, 3))
    coords = mol.atom_coords()
    for b in range(mol.nbas):
        centre[loc[b]:loc[b + 1]] = coords[mol.bas_atom(b)]
    return centre


def _density(case, mol, seed):
    '''(n_dm, nao, nao) or (nao, nao), numpy.  'delta': the change of a density
    between two SCF cycles, 1e-3 in every element; 'full': elements of order
    0.3 that decay with the distance of their centres as a density does.'''
    rng = np.random.default_rng(seed)
    shape = (case['n_dm'], mol.nao, mol.nao)
    g = rng.standard_normal(shape)
    if case['hermi'] == 1:
        g = (g + g.transpose(0, 2, 1)) / 2
    if case['density'] == 'delta':
        dm = 1e-3 * g
    else:
        r = _ao_centres(mol)
        d = np.linalg.norm(r[:, None, :] - r[None, :, :], axis=2)
        dm = .3 * g * np.exp(-d / 2.5)
    return dm if case['n_dm'] > 1 else dm[0]


def prepare(case, seed):
    if case['kind'] == 'scf':
        # one molecule per seed; everything else is the call's own work
        return dict(kind='scf', mol=_molecule(case, case['geom'] + 7919 * seed))
    mol = _molecule(case, case['geom'])
    dm = torch.as_tensor(_density(case, mol, seed), device='cuda')
    if case['kind'] == 'j_md':
        opt = j_engine._VHFOpt(mol, DIRECT_SCF_TOL).build()
    else:
        opt = jk._VHFOpt(mol, DIRECT_SCF_TOL).build()
    return dict(kind=case['kind'], mol=mol, dm=dm, opt=opt, hermi=case['hermi'])


def run(state):
    kind, mol = state['kind'], state['mol']
    if kind == 'scf':
        mf = RHF(mol)
        e_tot = mf.kernel()
        return dict(e_tot=e_tot, mo_energy=mf.mo_energy, dm=mf.dm)
    dm, opt = state['dm'], state['opt']
    if kind == 'jk':
        vj, vk = jk.get_jk(mol, dm, hermi=state['hermi'], vhfopt=opt)
        return dict(vj=vj, vk=vk)
    if kind == 'mixed':
        dms = opt.apply_coeff_C_mat_CT(dm[None])
        vj, vk = opt.get_jk(dms, state['hermi'], fp32_tol=FP32_TOL)
        return dict(vj=opt.apply_coeff_CT_mat_C(vj), vk=opt.apply_coeff_CT_mat_C(vk))
    if kind == 'rsh_k':
        return dict(vk=jk.get_k(mol, dm, hermi=1, vhfopt=opt, **RSH))
    if kind == 'j_md':
        return dict(vj=j_engine.get_j(mol, dm, hermi=1, vhfopt=opt))
    return dict(de=grad_rhf._jk_energy_per_atom(opt, dm))


# -- work -----------------------------------------------------------------
def _segments(mol):
    '''Shells in segments as the engine contracts them (primitives with
    exponents up to 0.3 on their own): (centre, l, exponents, coefficients).'''
    out = []
    for b in range(mol.nbas):
        es, cs = mol.bas_exp(b), mol.bas_ctr_coeff(b)[:, 0]
        parts = [np.where(es > .3)[0]] + [np.array([p]) for p in np.where(es <= .3)[0]]
        for p in parts:
            if len(p):
                out.append((mol.bas_coord(b), mol.bas_angular(b), es[p], np.abs(cs[p])))
    return out


def _quartets(mol, dmax, tol=DIRECT_SCF_TOL):
    '''{((li, pi), ...): estimated quartets with sqrt|(ij|ij)(kl|kl)| dmax > tol},
    from s-type estimates of the Schwarz factors.'''
    seg = _segments(mol)
    groups = sorted({(s[1], len(s[2])) for s in seg})
    pairs = {}
    for gi, a in enumerate(groups):
        for b in groups[:gi + 1]:
            A = [s for s in seg if (s[1], len(s[2])) == a]
            B = [s for s in seg if (s[1], len(s[2])) == b]
            ra, rb = np.array([s[0] for s in A]), np.array([s[0] for s in B])
            r2 = ((ra[:, None] - rb[None]) ** 2).sum(-1)
            q = np.zeros(r2.shape)
            for x in range(a[1]):
                ea, ca = (np.array([s[k][x] for s in A])[:, None] for k in (2, 3))
                for y in range(b[1]):
                    eb, cb = (np.array([s[k][y] for s in B])[None] for k in (2, 3))
                    p = ea + eb
                    q += (ca * cb / (4 * math.pi) * np.exp(-ea * eb / p * r2) *
                          (math.pi / p) ** 1.5 * (2. / math.pi) ** .5 * p ** .25)
            q = q[np.tril_indices(len(A))] if a == b else q.ravel()
            pairs[a, b] = np.sort(q[q > tol])
    keys = sorted(pairs)
    out = {}
    for m, ij in enumerate(keys):
        for kl in keys[:m + 1]:
            x, y = pairs[ij], pairs[kl]
            if len(x) and len(y):
                n = (len(y) - np.searchsorted(y, tol / (dmax * x))).sum()
                out[ij + kl] = float(n) * (.5 if ij == kl else 1.)
    return out


def _nc(l):
    return (l + 1) * (l + 2) // 2


def work(case):
    '''Bytes: density in, matrices out.  FLOPs of one estimated set of
    surviving quartets: per primitive quartet and root 3 per block element
    and 9 per element of the 2D tables, 4 per block element, density and
    matrix digested for each of the blocks of J (2) and of K (4); a gradient
    contracts three more tables.'''
    mol = _molecule(case, case['geom'])
    kind, n_dm = case['kind'], case['n_dm'] * (2 if case['hermi'] == 0 else 1)
    dmax = {'delta': 4e-3, 'full': 1.}[case['density']]
    blocks = {'rsh_k': 4, 'j_md': 2}.get(kind, 6)
    flops = 0.
    for key, n in _quartets(mol, dmax).items():
        ls, ps = [g[0] for g in key], [g[1] for g in key]
        nf = math.prod(_nc(l) for l in ls)
        g2 = (ls[0] + ls[1] + 1) * (ls[2] + ls[3] + 1)
        roots = sum(ls) // 2 + 1
        eri = math.prod(ps) * roots * (3 * nf + 9 * g2)
        if kind == 'rsh_k':
            eri *= 2            # full range and attenuated
        if kind == 'grad':
            eri *= 4
        flops += n * (eri + 2 * blocks * n_dm * nf)
    mats = case['n_dm'] * mol.nao ** 2 * 8
    nbytes = mats * {'rsh_k': 2, 'j_md': 2, 'grad': 1, 'scf': 2}.get(kind, 3)
    if kind == 'scf':
        flops *= 9              # cycles of a water cluster
    return dict(bytes=float(nbytes), flops=flops)


# -- 64-bit values of the small cases ---------------------------------------
def _powers(l):
    return [(x, y, l - x - y) for x in range(l, -1, -1) for y in range(l - x, -1, -1)]


def _harmonics(l):
    '''(2l+1, ncart) real solid harmonics in the Cartesian monomials, l <= 3;
    p in the order x, y, z.'''
    if l == 0:
        return [[.5 / math.sqrt(math.pi)]]
    if l == 1:
        s = math.sqrt(3. / (4 * math.pi))
        return [[s, 0, 0], [0, s, 0], [0, 0, s]]
    pi = math.pi
    if l == 2:      # xx xy xz yy yz zz
        a, b, c = math.sqrt(15 / (4 * pi)), math.sqrt(5 / (16 * pi)), math.sqrt(15 / (16 * pi))
        return [[0, a, 0, 0, 0, 0], [0, 0, 0, 0, a, 0], [-b, 0, 0, -b, 0, 2 * b],
                [0, 0, a, 0, 0, 0], [c, 0, 0, -c, 0, 0]]
    # xxx xxy xxz xyy xyz xzz yyy yyz yzz zzz
    a, b, c, d = (math.sqrt(x / (k * pi)) for x, k in ((35, 32), (105, 4), (21, 32), (7, 16)))
    return [[0, 3 * a, 0, 0, 0, 0, -a, 0, 0, 0], [0, 0, 0, 0, b, 0, 0, 0, 0, 0],
            [0, -c, 0, 0, 0, 0, -c, 0, 4 * c, 0], [0, 0, -3 * d, 0, 0, 0, 0, -3 * d, 0, 2 * d],
            [-c, 0, 0, -c, 0, 4 * c, 0, 0, 0, 0], [0, 0, b / 2, 0, 0, 0, 0, -b / 2, 0, 0],
            [a, 0, 0, -3 * a, 0, 0, 0, 0, 0, 0]]


def _boys(mmax, x):
    '''F_0..F_mmax(x): the series of the highest order and downward recursion,
    above x = 40 the closed form of F_0 and upward recursion.'''
    small = x < 40.
    xs = torch.where(small, x, torch.ones_like(x))
    term = torch.full_like(x, 1. / (2 * mmax + 1))
    s = term.clone()
    for k in range(1, 180):
        term = term * (2 * xs) / (2 * mmax + 2 * k + 1)
        s += term
    f = [None] * (mmax + 1)
    e = torch.exp(-xs)
    f[mmax] = s * e
    for m in range(mmax, 0, -1):
        f[m - 1] = (2 * xs * f[m] + e) / (2 * m - 1)
    xl = torch.where(small, torch.full_like(x, 40.), x)
    g = .5 * torch.sqrt(math.pi / xl) * torch.erf(torch.sqrt(xl))
    e = torch.exp(-xl)
    out = []
    for m in range(mmax + 1):
        out.append(torch.where(small, f[m], g))
        g = ((2 * m + 1) * g - e) / (2 * xl)
    return out


def _eri(mol, parts):
    '''(nao, nao, nao, nao) integrals of sum_parts weight * operator, with
    parts [(omega, weight)] of erf(omega r)/r (omega None: 1/r), by the
    McMurchie-Davidson scheme.'''
    dev = 'cuda' if torch.cuda.is_available() else 'cpu'
    shells = []         # centre, l, exponents, coefficients of one contraction
    for b in range(mol.nbas):
        for c in mol.bas_ctr_coeff(b).T:
            shells.append((mol.bas_coord(b), mol.bas_angular(b), mol.bas_exp(b), c))
    lmax = max(s[1] for s in shells)
    prims, pair_of = [], []
    pairs = [(i, j) for i in range(len(shells)) for j in range(i + 1)]
    for n, (i, j) in enumerate(pairs):
        for a, ca in zip(shells[i][2], shells[i][3]):
            for b, cb in zip(shells[j][2], shells[j][3]):
                prims.append(np.concatenate([[a, b, ca * cb], shells[i][0], shells[j][0]]))
                pair_of.append(n)
    t = torch.as_tensor(np.array(prims), device=dev)
    pair_of = np.array(pair_of)
    a, b = t[:, 0], t[:, 1]
    p = a + b
    A, B = t[:, 3:6], t[:, 6:9]
    P = (a[:, None] * A + b[:, None] * B) / p[:, None]
    K = t[:, 2] * torch.exp(-a * b / p * ((A - B) ** 2).sum(1))
    E = []              # E[d][i][j]: (n_prim_pairs, i + j + 1)
    for d in range(3):
        e = [[None] * (lmax + 1) for _ in range(lmax + 1)]
        e[0][0] = torch.ones_like(p)[:, None]

        def raised(x, shift):
            n = x.shape[1]
            y = torch.zeros((len(p), n + 1), dtype=p.dtype, device=dev)
            y[:, 1:] += x / (2 * p)[:, None]
            y[:, :n] += shift[:, None] * x
            y[:, :n - 1] += torch.arange(1, n, device=dev) * x[:, 1:]
            return y
        for i in range(lmax + 1):
            if i:
                e[i][0] = raised(e[i - 1][0], P[:, d] - A[:, d])
            for j in range(1, lmax + 1):
                e[i][j] = raised(e[i][j - 1], P[:, d] - B[:, d])
        E.append(e)
    herm = [h for n in range(2 * lmax + 1) for h in _powers(n)]
    at = {h: n for n, h in enumerate(herm)}
    harm = [torch.as_tensor(_harmonics(s[1]), dtype=torch.float64, device=dev) for s in shells]
    rows = []           # per shell pair: (functions, primitive pairs, Hermites)
    for n, (i, j) in enumerate(pairs):
        idx = torch.as_tensor(np.where(pair_of == n)[0], device=dev)
        ci, cj = _powers(shells[i][1]), _powers(shells[j][1])
        x = torch.zeros((len(ci), len(cj), len(idx), len(herm)), dtype=p.dtype, device=dev)
        for m, u in enumerate(ci):
            for q, v in enumerate(cj):
                ex, ey, ez = (E[d][u[d]][v[d]][idx] for d in range(3))
                for tx in range(ex.shape[1]):
                    for ty in range(ey.shape[1]):
                        for tz in range(ez.shape[1]):
                            x[m, q, :, at[tx, ty, tz]] += (K[idx] * ex[:, tx] * ey[:, ty] *
                                                           ez[:, tz])
        x = torch.tensordot(harm[j], torch.tensordot(harm[i], x, 1), ([1], [1]))
        rows.append((idx, x.transpose(0, 1).reshape(-1, len(idx), len(herm))))
    sign = torch.as_tensor([(-1.) ** sum(h) for h in herm], device=dev, dtype=torch.float64)
    nf = [len(h) for h in harm]
    loc = np.concatenate([[0], np.cumsum(nf)])
    nao = int(loc[-1])
    n_fn = sum(len(r[1]) for r in rows)
    ket = torch.zeros((n_fn, len(p), len(herm)), dtype=torch.float64, device=dev)
    ij = []
    pos = 0
    for (i, j), (idx, x) in zip(pairs, rows):
        ket[pos:pos + len(x), idx] = x * sign
        ij += [(loc[i] + m, loc[j] + q) for m in range(nf[i]) for q in range(nf[j])]
        pos += len(x)
    ket = ket.reshape(n_fn, -1)
    tri = torch.empty((n_fn, n_fn), dtype=torch.float64, device=dev)
    pos = 0
    for (i, j), (idx, x) in zip(pairs, rows):
        L = 2 * lmax + shells[i][1] + shells[j][1]
        d = P[idx][:, None] - P[None]
        pq = p[idx][:, None] + p[None]
        alpha0 = p[idx][:, None] * p[None] / pq
        pref = 2 * math.pi ** 2.5 / (p[idx][:, None] * p[None] * torch.sqrt(pq))
        r0 = [0.] * (L + 1)
        for omega, weight in parts:
            al = alpha0 if omega is None else alpha0 * omega ** 2 / (alpha0 + omega ** 2)
            c = weight * pref * torch.sqrt(al / alpha0)
            for m, f in enumerate(_boys(L, al * (d ** 2).sum(-1))):
                r0[m] = r0[m] + c * (-2 * al) ** m * f
        level = {(0, 0, 0): r0[L]}
        for m in range(L - 1, -1, -1):
            new = {(0, 0, 0): r0[m]}
            for n in range(1, L - m + 1):
                for h in _powers(n):
                    k = next(k for k in range(3) if h[k])
                    g = list(h)
                    g[k] -= 1
                    v = d[..., k] * level[tuple(g)]
                    if g[k]:
                        f = g[k]
                        g[k] -= 1
                        v = v + f * level[tuple(g)]
                    new[h] = v
            level = new
        acc = torch.zeros((len(x), len(p), len(herm)), dtype=torch.float64, device=dev)
        for m, h in enumerate(herm):
            if sum(h) > shells[i][1] + shells[j][1]:
                continue
            for q, g in enumerate(herm):
                acc[:, :, q] += x[:, :, m] @ level[h[0] + g[0], h[1] + g[1], h[2] + g[2]]
        tri[pos:pos + len(x)] = acc.reshape(len(x), -1) @ ket.T
        pos += len(x)
    ij = np.array(ij)
    full = np.zeros((nao, nao), dtype=np.int64)
    full[ij[:, 0], ij[:, 1]] = np.arange(n_fn)
    full = np.tril(full) + np.tril(full, -1).T
    k = torch.as_tensor(full.ravel(), device=dev)
    return tri[k][:, k].reshape(nao, nao, nao, nao)


def exact(case, seed):
    if case['kind'] not in ('jk', 'mixed', 'rsh_k', 'j_md') or case['basis'] == TZVP_G:
        return None
    if case['system'] != 'water' or case['n'] > (2 if case['basis'] == SVP else 1):
        return None
    mol = _molecule(case, case['geom'])
    dm = _density(case, mol, seed)
    if case['kind'] == 'rsh_k':
        eri = _eri(mol, [(None, RSH['sr_factor']), (RSH['omega'],
                                                    RSH['lr_factor'] - RSH['sr_factor'])])
    else:
        eri = _eri(mol, [(None, 1.)])
    dms = torch.as_tensor(dm, device=eri.device).reshape(-1, mol.nao, mol.nao)
    vj = torch.einsum('ijkl,nlk->nij', eri, dms).reshape(dm.shape)
    vk = torch.einsum('ijkl,njk->nil', eri, dms).reshape(dm.shape)
    if case['kind'] == 'rsh_k':
        return dict(vk=vk)
    if case['kind'] == 'j_md':
        return dict(vj=vj)
    if case['kind'] == 'mixed':
        vj, vk = vj[None], vk[None]
    return dict(vj=vj, vk=vk)
