"""The four-step phi kernels and the fused cross product in small tiles (a launch
of few workgroups) and in large ones: the same bits.  A flow that does not depend
on z has the same advection term in a kit of 2 slices (small tiles) and in one of
512 (large tiles): its z transforms add and subtract equal numbers, which is exact."""
import numpy as np
import pytest

import _cases as C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nph', [16, 32, 64, 128])
def test_same_bits(nph):
    import mlegs_amd as M
    print('tiles', nph, flush=True)
    out = []
    for nz in (2, 512):
        p = C.params(C.C1, nr=66, np=2 * nph, nz=nz, nrchop=62, npchop=nph + 1, nzchop=nz // 2 + 1, ell=1.4)
        tfm = M.Kit(p)
        f = []
        for i in range(2):
            e = np.zeros(tfm.dims, dtype=np.complex128)
            c = C.spectral((p.nr + 3, nph + 1, 2), C.params(p.__dict__, nz=2, nzchop=2), 80 + i)
            e[:, :, 0] = c[:, :, 0]
            f.append(M.Scalar(tfm).upload(e, space='FFF'))
        uz = M.Scalar(tfm)
        n, m = M.Scalar(tfm), M.Scalar(tfm)
        M.advection_rhs(f[0], f[1], n, m, uz, tfm)
        assert not np.any(n.e[:, :, 1:]) and not np.any(m.e[:, :, 1:])
        out.append((n.e[:, :, 0].copy(), m.e[:, :, 0].copy()))
        tfm.close()
    for a, b in zip(*out):
        assert np.any(a) and np.array_equal(a, b)
