"""The four-step FFT kernels run small tiles where a launch has few workgroups
and large ones elsewhere: phi and z transforms at both, with ragged row counts,
and the fused cross product at both, against the oracle.

Tolerance of the transforms: 5 eps log2(512) = 5e-15, doubled.  advection_rhs:
test_gpu_parity's 1e-10."""
import numpy as np
import pytest

import _cases as C

pytestmark = pytest.mark.gpu


def rel_err(a, b):
    return np.linalg.norm((a - b).ravel()) / max(np.linalg.norm(b.ravel()), 1e-300)


@pytest.mark.parametrize('n', (16, 32, 64, 128))
@pytest.mark.parametrize('many', (2, 540))
def test_phi_and_z(n, many):
    import mlegs_amd as M
    from oracle import kit as K, scalar_ops as so
    for np_, nz, pairs in ((2 * n, many, (('PPP', 'PFP'), ('PFP', 'PPP'))),
                           (2 * many, n, (('FFP', 'FFF'), ('FFF', 'FFP')))):
        print('length', n, 'grid', np_, nz, flush=True)
        p = C.params(C.C1, nr=18, np=np_, nz=nz, nrchop=18, npchop=3, nzchop=nz // 2 + 1)
        tfm, okit = M.Kit(p), K.Kit3D(p)
        rng = np.random.default_rng(n)
        for a, b in pairs:
            e = rng.standard_normal(tfm.dims) + 1j * rng.standard_normal(tfm.dims)
            g, o = C.pair(tfm, okit, e, a)
            M.trans(g, b, tfm)
            so.trans(o, b, okit)
            assert rel_err(g.e, o.e) < 1e-14, (a, b, np_, nz)
        tfm.close()


@pytest.mark.parametrize('n', (16, 32, 64, 128))
@pytest.mark.parametrize('nz', (2, 512))
def test_cross_product(n, nz):
    import mlegs_amd as M
    from oracle import kit as K, scalar_ops as so, vortex as V
    print('cross', 2 * n, nz, flush=True)
    p = C.params(C.C1, nr=18, np=2 * n, nz=nz, nrchop=17, npchop=9, nzchop=min(nz // 2 + 1, 9), ell=1.4)
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
