"""The phi and z transforms at every kind of length (one, two, three and four
register groups, odd lengths, the four-step powers of two, lengths past 256)
and the fused cross product at non-power-of-two lengths, against the oracle.

Tolerance of the transforms: a mixed-radix FFT's norm-wise error is below
5 eps log2(512) = 5e-15; 1e-14 is twice that.  advection_rhs: test_gpu_parity's
1e-10 (its grids are of that size)."""
import numpy as np
import pytest

import _cases as C

pytestmark = pytest.mark.gpu

LENGTHS = (1, 2, 3, 5, 6, 8, 9, 10, 12, 15, 16, 18, 20, 25, 27, 32, 45, 54, 64, 75, 81, 96, 125, 128, 162, 200, 216,
           243, 250, 256, 320, 375, 400, 486, 500, 512)


def rel_err(a, b):
    return np.linalg.norm((a - b).ravel()) / max(np.linalg.norm(b.ravel()), 1e-300)


@pytest.mark.parametrize('n', LENGTHS)
def test_phi_and_z(n):
    import mlegs_amd as M
    from oracle import kit as K, scalar_ops as so
    print('length', n, flush=True)
    # n packed points in phi (np = 2 n), and n slices in z where the kit takes them
    nz = n if n % 2 == 0 else 1
    for np_, nz in ((2 * n, 2), (2, nz)):
        p = C.params(C.C1, nr=10, np=np_, nz=nz, nrchop=10, npchop=min(np_ // 2 + 1, 3), nzchop=nz // 2 + 1)
        tfm, okit = M.Kit(p), K.Kit3D(p)
        rng = np.random.default_rng(n)
        for a, b in (('PPP', 'PFP'), ('PFP', 'PPP'), ('FFP', 'FFF'), ('FFF', 'FFP')):
            e = rng.standard_normal(tfm.dims) + 1j * rng.standard_normal(tfm.dims)
            g, o = C.pair(tfm, okit, e, a)
            M.trans(g, b, tfm)
            so.trans(o, b, okit)
            assert rel_err(g.e, o.e) < 1e-14, (a, b, np_, nz)
        tfm.close()


@pytest.mark.parametrize('np_,nz', [(18, 10), (30, 6), (48, 32), (100, 4), (8, 18)])
def test_cross_product(np_, nz):
    import mlegs_amd as M
    from oracle import kit as K, scalar_ops as so, vortex as V
    print('cross', np_, nz, flush=True)
    p = C.params(C.C1, nr=34, np=np_, nz=nz, nrchop=33, npchop=np_ // 2 + 1, nzchop=nz // 2 + 1, ell=1.4)
    tfm, okit = M.Kit(p), K.Kit3D(p)
    (gpsi, opsi), (gchi, ochi) = C.qvortex(tfm, okit, p, amp=0.5)
    ub = C.physical(tfm.dims, p, 31)
    guz = M.Scalar(tfm).upload(ub, space='PPP')
    ouz = so.Scalar(okit, 'PPP')
    ouz.e = ub.copy()
    gnp, gnc = M.Scalar(tfm), M.Scalar(tfm)
    M.advection_rhs(gpsi, gchi, gnp, gnc, guz, tfm)
    onp, onc = V.advection_rhs(opsi, ochi, ouz, okit)
    assert rel_err(gnp.e, onp.e) < 1e-10 and rel_err(gnc.e, onc.e) < 1e-10
    tfm.close()
