"""The vortex step's SVV filter takes the value at infinity off on the same pass:
against svv_filter and zeroat1 one after another, on kits whose column 0 has fewer
rows than, as many as and more than a workgroup has threads, with the filter engaged.

Tolerance: the filter's two sums run over other ranges there (the de-aliased modes are
left out), so the gain may differ by a few eps; exp(-strength ..) <= 1 passes that
on as such, and zeroat1's correction adds nr eps of the column: 1e-12."""
import numpy as np
import pytest

import _cases as C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nr,np_,nz', [(30, 16, 12), (256, 8, 2), (270, 12, 1), (48, 64, 18)])
def test_filter_and_zeroat1(nr, np_, nz):
    import mlegs_amd as M
    print('svv zeroat1', nr, np_, nz, flush=True)
    p = C.params(C.SMALL, nr=nr, np=np_, nz=nz, nrchop=nr, npchop=np_ // 2 + 1, nzchop=nz // 2 + 1, is_svv=True)
    tfm = M.Kit(p)
    f = [M.Scalar(tfm).upload(C.spectral(tfm.dims, p, 70 + i, decay=1e4), space='FFF', ln=0.1 * (i + 1))
         for i in range(6)]
    for s in f:
        M.dealias(s, tfm)
    uz = M.Scalar(tfm).upload(C.physical(tfm.dims, p, 7), space='PPP')
    run = M.VortexRun(tfm, f[0], f[1], uz)
    for nm, s in zip(('psi', 'chi', 'nlpsi', 'nlchi', 'nlpsi_prev', 'nlchi_prev'), f):
        run.field(nm).assign(s)
    run.step(1, check=False)
    for s, n, n_p, nm in ((f[0], f[2], f[4], 'psi'), (f[1], f[3], f[5], 'chi')):
        M.abcn(s, s.copy(), n, n_p, p.dt, tfm)
        M.dealias(s, tfm)
        before = s.e
        assert M.svv_filter(s, tfm, 0.0) > 0.0 and not np.array_equal(before, s.e)
        M.zeroat1(s, tfm)
        e = run.field(nm).e
        assert np.linalg.norm((e - s.e).ravel()) < 1e-12 * np.linalg.norm(s.e.ravel())
        assert run.field(nm).ln == s.ln
    tfm.close()
