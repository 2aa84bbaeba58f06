"""Fields whose memory another field held before: new fields are zero, live ones
keep their values, over kits of two sizes and two threads, through more fields
than are kept; and work of another stream on a field's memory, issued before the
field ended, is done before a new field holds that memory."""
import gc
import threading

import numpy as np
import pytest

import _cases as C

pytestmark = pytest.mark.gpu


def _churn(M, tfm, seed, rounds, errs):
    try:
        rng = np.random.default_rng(seed)
        keep = []
        for k in range(rounds):
            f = M.Scalar(tfm, 'FFF')
            assert f.space == 'FFF' and f.ln == 0.0
            if k % 9 == 0:
                assert not np.any(f.e)
            a = np.zeros(tfm.dims, dtype=np.complex128)
            a[:4] = rng.standard_normal() + 2.0 + 1j
            f.upload(a, space='FFF', ln=float(k + 1))
            if k % 5 == 0:
                g = f.copy()
                keep.append((g, a, float(k + 1)))
                if len(keep) > 6:
                    keep.pop(0)
        for g, a, ln in keep:
            assert np.array_equal(g.e, a) and g.ln == ln and g.space == 'FFF'
    except Exception as e:  # noqa: BLE001 - reported by the main thread
        errs.append(e)


def test_reused_memory():
    import mlegs_amd as M
    kits = [M.Kit(C.params(C.SMALL)), M.Kit(C.params(C.POW2))]
    errs = []
    th = [threading.Thread(target=_churn, args=(M, t, i, 90, errs)) for i, t in enumerate(kits)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errs, errs
    gc.collect()
    for t in kits:
        t.close()


def test_other_stream_first():
    """A second context's stream, behind some milliseconds of work of its own,
    reads a field of the first; the field ends before that, and no field the
    first makes meanwhile changes what is read."""
    import mlegs_amd as M
    p = C.params(C.POW2)
    tfm, other = M.Kit(p), M.Kit(p)
    busy, got = M.Scalar(other, 'FFF'), M.Scalar(other)
    a = np.full(tfm.dims, 3.0 + 0.0j)
    for _ in range(3):
        f = M.Scalar(tfm, 'FFF').upload(a, space='FFF')
        for _ in range(300):
            M.trans(busy, 'PPP', other)
            M.trans(busy, 'FFF', other)
        other._check(other.lib.mlx_field_copy(other.ctx, got.h, f.h))
        del f
        for _ in range(2):
            new = [M.Scalar(tfm) for _ in range(40)]
            del new
        assert np.array_equal(got.e, a)
    tfm.close()
    other.close()
