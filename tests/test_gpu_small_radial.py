"""advection_rhs on the smallest radial grids, whose columns are shorter than a
line of FP32 radial pairs: lengths of the phi transform with and without
four-step kernels, against the oracle.

Tolerances, norm-wise relative, of psi and of chi's Laplacian (the projection's
own products): FP64 1e-10 (test_gpu_parity.py).  FP32: the velocity and the
vorticity carry their operands' and sums' rounding, at most 6 x 2^-24 for sums of
up to four terms, their product twice that, and the projection's own sums as
much again: 1e-6; the differences of the D and T tables cancel by up to a factor
of ten: 1e-5."""
import numpy as np
import pytest

import _cases as C

pytestmark = pytest.mark.gpu


def rel_err(a, b):
    return np.linalg.norm((a - b).ravel()) / max(np.linalg.norm(b.ravel()), 1e-300)


@pytest.mark.parametrize('nr,np_,nz', [(4, 12, 4), (2, 12, 4), (4, 10, 2), (4, 32, 4), (6, 12, 4)])
@pytest.mark.parametrize('prec,tol', [('FP64', 1e-10), ('FP32', 1e-5), ('BF16X3', 1e-5)])
def test_advection_rhs(nr, np_, nz, prec, tol):
    import mlegs_amd as M
    from oracle import kit as K, scalar_ops as so, vortex as V
    print('small radial', nr, np_, nz, prec, flush=True)
    p = C.params(C.C1, nr=nr, np=np_, nz=nz, nrchop=nr, npchop=np_ // 2 + 1, nzchop=nz // 2 + 1, ell=1.3)
    tfm, okit = M.Kit(p, precision=getattr(M, 'PREC_' + prec)), K.Kit3D(p)
    gpsi, opsi = C.pair(tfm, okit, C.spectral(tfm.dims, p, 5), 'FFF')
    gchi, ochi = C.pair(tfm, okit, C.spectral(tfm.dims, p, 6), 'FFF')
    guz, ouz = C.pair(tfm, okit, C.physical(tfm.dims, p, 7), 'PPP')
    gn, gc = M.Scalar(tfm), M.Scalar(tfm)
    M.advection_rhs(gpsi, gchi, gn, gc, guz, tfm)
    on, oc = V.advection_rhs(opsi, ochi, ouz, okit)
    assert rel_err(gn.e, on.e) < tol
    M.del2(gc, tfm)
    so.del2(oc, okit)
    assert rel_err(gc.e, oc.e) < tol
    tfm.close()
