"""A field that another kit's context ends: its memory keeps its own size, so a
field of the larger kit made later gets a block of its own size (zero, and no
live field of the smaller kit changes)."""
import numpy as np
import pytest

import _cases as C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('ends', ['larger', 'smaller'])
def test_ended_by_another_kit(ends):
    import mlegs_amd as M
    print('ended by the', ends, 'kit', flush=True)
    small, large = M.Kit(C.params(C.SMALL)), M.Kit(C.params(C.ODD))
    own, other = (small, large) if ends == 'larger' else (large, small)
    live = [M.Scalar(small).upload(np.full(small.dims, k + 1.0j), space='FFF') for k in range(8)]
    for _ in range(80):  # past the number of blocks that one wait serves
        f = M.Scalar(own, 'FFF')
        other._check(other.lib.mlx_field_destroy(other.ctx, f.h))
        f.h = None
    new = [M.Scalar(large) for _ in range(70)]
    for f in new[::9]:
        assert not np.any(f.e)
    for k, f in enumerate(live):
        assert np.array_equal(f.e, np.full(small.dims, k + 1.0j))
    del new, live
    small.close()
    large.close()
