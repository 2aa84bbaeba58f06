"""Which arithmetic vec2tp's projection takes.

A radial chopping offset on chi, whose solve reads three rows past the chopped
ones: past 256 radial points every precision forms them in FP64, against the
oracle (test_gpu_parity's 1e-10; chi through its Laplacian, the projection's own
product).  And the projection's own precision set to FP64 where the context's is
lower: every column is formed in FP64."""
import numpy as np
import pytest

import _cases as C

pytestmark = pytest.mark.gpu


def rel_err(a, b):
    return np.linalg.norm((a - b).ravel()) / max(np.linalg.norm(b.ravel()), 1e-300)


@pytest.mark.parametrize('prec', ['FP64', 'FP64_MFMA', 'FP32', 'BF16X3'])
def test_offset_past_256_points(prec, monkeypatch):
    import mlegs_amd as M
    from oracle import kit as K, scalar_ops as so
    print('offset past 256', prec, flush=True)
    p = C.params(C.C1, nr=258, np=8, nz=6, nrchop=256, npchop=5, nzchop=4, ell=1.3)
    tfm, okit = M.Kit(p, precision=getattr(M, 'PREC_' + prec)), K.Kit3D(p)
    v = [C.pair(tfm, okit, C.physical(tfm.dims, p, 60 + i), 'PPP') for i in range(3)]
    psi, chi = M.Scalar(tfm), M.Scalar(tfm)
    chi.chop_offset(3)
    M.vec2tp(*(g for g, _ in v), psi, chi, tfm)
    solve = so.idel2_proln

    def over_offset(s, kit):  # the solve runs over the rows of chi's own offset
        s.chop_offset(3)
        solve(s, kit)
    monkeypatch.setattr(so, 'idel2_proln', over_offset)
    opsi, ochi = so.vec2tp(*(o for _, o in v), okit)
    assert rel_err(psi.e, opsi.e) < 1e-10
    M.del2(chi, tfm)
    so.del2(ochi, okit)
    assert rel_err(chi.e, ochi.e) < 1e-10
    tfm.close()


@pytest.mark.parametrize('cfg', ['C1', 'SMALL', 'ODD'])
@pytest.mark.parametrize('ctx', ['FP32', 'BF16X3'])
def test_fp64_projection_of_a_reduced_context(cfg, ctx):
    """The projection and the transform before it set to FP64: the result of a
    context in FP64, bit for bit, column 0 included."""
    import mlegs_amd as M
    print('fp64 projection', cfg, ctx, flush=True)
    p = C.params(getattr(C, cfg))
    out = []
    for prec in ('FP64', ctx):
        tfm = M.Kit(p, precision=getattr(M, 'PREC_' + prec))
        if prec != 'FP64':
            tfm.set_stage_precision(M.STAGE_UP, M.PREC_FP64)
            tfm.set_stage_precision(M.STAGE_PROJ, M.PREC_FP64)
        v = [M.Scalar(tfm).upload(C.physical(tfm.dims, p, 70 + i), space='PPP') for i in range(3)]
        psi, chi = M.Scalar(tfm), M.Scalar(tfm)
        M.vec2tp(*v, psi, chi, tfm)
        out.append((psi.e, psi.ln, chi.e, chi.ln))
        tfm.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
