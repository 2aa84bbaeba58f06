"""The hyperviscous solve at several workgroups per column, against the oracle,
and psi and chi solved in one launch by the vortex step against one field at a
time (abcn), bit for bit: the same operations in the same order.

ihelmp against the oracle: test_gpu_parity's tolerances (1e-6, residual 1e-8)."""
import numpy as np
import pytest

import _cases as C

pytestmark = pytest.mark.gpu


def rel_err(a, b):
    return np.linalg.norm((a - b).ravel()) / max(np.linalg.norm(b.ravel()), 1e-300)


@pytest.mark.parametrize('power,alpha,beta', [(4, 2.0e3, -0.8), (6, -55.0, 1.5), (8, 1.0e6, -0.5)])
def test_ihelmp_many_slices(power, alpha, beta):
    import mlegs_amd as M
    from oracle import kit as K, scalar_ops as so
    print('ihelmp', power, flush=True)
    p = C.params(C.C1, nr=26, np=8, nz=80, nrchop=25, npchop=5, nzchop=41)
    tfm, okit = M.Kit(p), K.Kit3D(p)
    g, o = C.pair(tfm, okit, C.spectral(tfm.dims, p, 23), 'FFF', ln=0.37)
    s0 = o.copy()
    M.ihelmp(g, power, alpha, beta, tfm)
    so.ihelmp(o, power, alpha, beta, okit)
    assert rel_err(g.e, o.e) < 1e-6
    back = o.copy()
    back.e, back.ln = g.e.copy(), g.ln
    so.helmp(back, power, alpha, beta, okit)
    assert rel_err(back.e, s0.e) < 1e-8
    tfm.close()


@pytest.mark.parametrize('nr,np_,nz,power', [(26, 8, 80, 8), (32, 12, 18, 6), (16, 24, 6, 4), (34, 16, 2, 8),
                                             (20, 10, 64, 4)])
def test_pair_is_single(nr, np_, nz, power):
    import mlegs_amd as M
    print('pair', nr, np_, nz, power, flush=True)
    p = C.params(C.C1, nr=nr, np=np_, nz=nz, nrchop=nr, npchop=np_ // 2 + 1, nzchop=nz // 2 + 1, hyperpow=power,
                 hypervisc=1e-7)
    tfm = M.Kit(p)
    (psi, chi, n1, n2, n1p, n2p) = [M.Scalar(tfm).upload(C.spectral(tfm.dims, p, 40 + i), space='FFF',
                                                         ln=0.1 * (i + 1)) for i in range(6)]
    for s in (psi, chi, n1, n2, n1p, n2p):
        M.dealias(s, tfm)
    uz = M.Scalar(tfm).upload(C.physical(tfm.dims, p, 7), space='PPP')
    run = M.VortexRun(tfm, psi, chi, uz)
    for nm, f in (('psi', psi), ('chi', chi), ('nlpsi', n1), ('nlchi', n2), ('nlpsi_prev', n1p), ('nlchi_prev', n2p)):
        run.field(nm).assign(f)
    run.step(1, check=False)
    got = [(run.field(nm).e, run.field(nm).ln) for nm in ('psi', 'chi')]
    for s, n, n_p, (e, ln) in ((psi, n1, n1p, got[0]), (chi, n2, n2p, got[1])):
        sp = s.copy()
        M.abcn(s, sp, n, n_p, p.dt, tfm)
        M.dealias(s, tfm)
        M.zeroat1(s, tfm)
        assert np.array_equal(s.e, e)
        assert s.ln == ln
    tfm.close()
