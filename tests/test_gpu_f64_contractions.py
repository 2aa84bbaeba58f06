"""The FP64 MFMA contractions (legendre_f64.hip) at the edges of their tiles
against the oracle: rows just below, at and past 16- and 64-row tiles, an odd
number of nodes per half, radial grids past 256 points (several row splits),
one axial slice, ragged slice tiles, columns that leave XCD groups of eight,
and the projection of a result with a radial chopping offset, which takes the
general kernel.

Tolerances: the FP64 ones of test_gpu_parity.py (transforms 1e-12, vec2tp
1e-10), norm-wise relative.  chi is compared through its Laplacian, that is on
the projection's own product: the kappa = 0 systems solved for it have
condition numbers of 1e6 to 1e12 at these radial sizes, so chi itself is fixed
to 1e-10 by no FP64 arithmetic, while the residual of the banded solves is
rounding times |A| |x| row by row, small where the coefficients have decayed."""
import numpy as np
import pytest

import _cases as C

pytestmark = pytest.mark.gpu

# nr, np, nz, nrchop, npchop, nzchop
KITS = {
    'nodes17': (34, 16, 10, 33, 9, 6),
    'rows63': (130, 20, 18, 125, 11, 10),
    'rows65': (130, 32, 32, 130, 17, 17),
    'one_slice': (98, 24, 1, 97, 13, 1),
    'past256': (258, 8, 6, 257, 5, 4),
    'splits': (390, 6, 4, 386, 3, 3),
    'wide': (66, 64, 40, 64, 33, 21),
}


def rel_err(a, b):
    return np.linalg.norm((a - b).ravel()) / max(np.linalg.norm(b.ravel()), 1e-300)


@pytest.fixture(scope='module', params=list(KITS))
def setup(request):
    import mlegs_amd as M
    from oracle import kit as K
    nr, np_, nz, a, b, d = KITS[request.param]
    p = C.params(C.C1, nr=nr, np=np_, nz=nz, nrchop=a, npchop=b, nzchop=d, ell=1.3)
    return request.param, p, M.Kit(p), K.Kit3D(p)


def test_transforms(setup):
    import mlegs_amd as M
    from oracle import scalar_ops as so
    name, p, tfm, okit = setup
    print('transforms', name, flush=True)
    g, o = C.pair(tfm, okit, C.spectral(tfm.dims, p, 3, decay=16.0), 'FFF', ln=0.4)
    M.trans(g, 'PPP', tfm)
    so.trans(o, 'PPP', okit)
    cols = max(1, p.np // 2)
    assert rel_err(g.e[:p.nr, :cols], o.e[:p.nr, :cols]) < 1e-12
    M.trans(g, 'FFF', tfm)
    so.trans(o, 'FFF', okit)
    assert rel_err(g.e, o.e) < 1e-12


@pytest.mark.parametrize('offset', [0, 3])
def test_projection(setup, offset, monkeypatch):
    import mlegs_amd as M
    from oracle import scalar_ops as so
    name, p, tfm, okit = setup
    print('projection', name, offset, flush=True)
    (gpsi, opsi), (gchi, ochi) = C.qvortex(tfm, okit, p, amp=1e-2)
    v = [M.Scalar(tfm) for _ in range(3)]
    M.tp2vec(gpsi, gchi, *v, tfm)
    ov = so.tp2vec(opsi, ochi, okit)
    psi, chi = M.Scalar(tfm), M.Scalar(tfm)
    chi.chop_offset(offset)
    M.vec2tp(*v, psi, chi, tfm)
    if offset:  # the result is solved over the rows of chi's own offset
        solve = so.idel2_proln

        def over_offset(s, kit):
            s.chop_offset(offset)
            solve(s, kit)
        monkeypatch.setattr(so, 'idel2_proln', over_offset)
    opsi2, ochi2 = so.vec2tp(*ov, okit)
    assert rel_err(psi.e, opsi2.e) < 1e-10
    M.del2(chi, tfm)
    so.del2(ochi2, okit)
    assert rel_err(chi.e, ochi2.e) < 1e-10


def test_projection_paths_agree(setup):
    """psi (which no solve follows) from the MFMA projection and from the
    general one, which an offset on chi selects: bit for bit."""
    import mlegs_amd as M
    name, p, tfm, okit = setup
    print('projection paths', name, flush=True)
    v = [M.Scalar(tfm).upload(C.physical(tfm.dims, p, i), space='PPP') for i in range(3)]
    psi = []
    for offset in (0, 3):
        a, b = M.Scalar(tfm), M.Scalar(tfm)
        b.chop_offset(offset)
        M.vec2tp(*v, a, b, tfm)
        psi.append(a.e)
    assert np.array_equal(psi[0], psi[1])
