"""abcn's copy of N into N_p rides on its right-hand side; where a field is given
twice it does not.  Both against the three operations one after another (the
step with other fields, then s_p <- s, then nl_p <- nl), bit for bit."""
import numpy as np
import pytest

import _cases as C

pytestmark = pytest.mark.gpu

NAMES = ('s', 's_p', 'nl', 'nl_p')
# which of the four arguments share a field
SHARED = [(), ('s', 'nl'), ('s', 'nl_p'), ('s_p', 'nl'), ('s_p', 'nl_p'), ('nl', 'nl_p'), ('s', 's_p')]


@pytest.mark.parametrize('cfg', [C.SMALL, dict(C.ODD, nz=1, nzchop=1), dict(C.POW2, nr=130, nrchop=127)],
                         ids=['small', 'polar', 'tall'])
@pytest.mark.parametrize('shared', SHARED, ids=lambda s: '='.join(s) or 'distinct')
def test_previous_terms(cfg, shared):
    import mlegs_amd as M
    print('abcn', shared, cfg['nr'], cfg['nz'], flush=True)
    p = C.params(cfg)
    tfm = M.Kit(p)
    new = lambda i: M.Scalar(tfm).upload(C.spectral(tfm.dims, p, 60 + i), space='FFF', ln=0.1 * i - 0.2)
    f = {n: new(i) for i, n in enumerate(NAMES)}
    if shared:
        f[shared[1]] = f[shared[0]]
    # the reference order on copies: the step leaves its first argument as s
    s, n, n_p = f['s'].copy(), f['nl'].copy(), f['nl_p'].copy()
    M.abcn(s, s.copy(), n, n_p, p.dt, tfm)
    want = {k: v.copy() for k, v in f.items()}
    for a, b in ((shared,) if shared else ()):
        want[b] = want[a]
    want['s'].assign(s)
    want['s_p'].assign(want['s'])
    want['nl_p'].assign(want['nl'])
    M.abcn(f['s'], f['s_p'], f['nl'], f['nl_p'], p.dt, tfm)
    for k in NAMES:
        assert np.array_equal(f[k].e, want[k].e), k
        assert f[k].ln == want[k].ln and f[k].space == want[k].space, k
    tfm.close()
