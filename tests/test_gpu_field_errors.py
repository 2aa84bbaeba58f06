"""A copy whose launch the runtime refuses (the stream's graph recording has been
broken off by a call that is not allowed in it) reports it.  In a process of its
own: the runtime leaves such a stream unusable."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.gpu

CODE = r'''
import ctypes, os, sys
sys.path[:0] = ['.', 'tests']
import _cases as C
import mlegs_amd as M
from mlegs_amd import _lib
lib = _lib.load()
p = C.params(C.SMALL)
ps = M._params_struct(p)
stream, graph, ctx = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
assert lib.hipStreamCreate(ctypes.byref(stream)) == 0
assert lib.mlx_ctx_create(ctypes.byref(ps), 0, stream, ctypes.byref(ctx)) == 0
assert lib.mlx_kit_init(ctx) == 0
tfm = M.Kit(p, _handle=ctx)
a, b = M.Scalar(tfm), M.Scalar(tfm)
b.upload(C.spectral(tfm.dims, p, 3), space='FFF')
assert lib.mlx_sync(ctx) == 0
assert lib.hipStreamBeginCapture(stream, 2) == 0
assert lib.hipStreamSynchronize(stream) != 0  # not allowed there: the recording is void
rc = lib.mlx_field_copy(ctx, a.h, b.h)
lib.hipStreamEndCapture(stream, ctypes.byref(graph))
print('copy', rc, 'hip error', _lib.MLX_E_HIP, flush=True)
os._exit(0 if rc == _lib.MLX_E_HIP else 1)
'''


def test_refused_copy_is_reported():
    r = subprocess.run([sys.executable, '-c', CODE], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
