"""Device memory of a kit past 256 radial points, where every contraction runs
in FP64: the FP32 tables of the contraction kernels are not made."""
import ctypes

import pytest

import _cases as C

pytestmark = pytest.mark.gpu


def _free(lib):
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_no_fp32_contraction_tables():
    import mlegs_amd as M
    p = C.params(C.C1, nr=512, np=256, nz=1, nrchop=512, npchop=129, nzchop=1)
    nrh, ne, nt, pitch = p.nr // 2, p.nrchop + 14, p.nrchop + 3, 256
    relaid = p.npchop * 2 * nrh * pitch           # one table, rows of one parity padded to 64
    plain = p.npchop * nrh * (ne + 3 * nt)        # Legendre table and V, D, T
    want = 12 * plain + 8 * 4 * relaid            # plain ones in FP64 and FP32, relaid ones in FP64
    tfm = M.Kit(C.params(C.SMALL))  # the library's own first use; its end gives back kept field memory
    tfm.close()
    before = _free(tfm.lib)
    tfm = M.Kit(p)
    used = before - _free(tfm.lib)
    print('kit of %.0f MB, tables %.0f MB' % (used / 1e6, want / 1e6), flush=True)
    # 4 x 4 relaid bytes more with the FP32 tables; allocations are padded
    assert want <= used < want + 8 * relaid
    tfm.close()
