"""Which way a field is copied (csrc/capi.hip, fcopy), on the CPU with the launch
and the runtime's copy replaced: a kernel reads another device's memory only where
peer access is on, which the runtime's copy does not need."""
import os
import subprocess

from mlegs_amd import build

DRIVER = r'''
#include "CAPI_SOURCE"
#include <cstdio>
static int kernels = 0, copies = 0;
extern "C" {
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *,
                           int *) {}
void __hipUnregisterFatBinary(void **) {}
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return ++copies, hipSuccess; }
}
namespace mlx {
void k_copy_field(mlx_ctx *, double2 *, const double2 *, double *, const double *) { ++kernels; }
}
int main() {
  mlx_ctx c;
  c.nelem = 1000;
  mlx_field d, s;
  int bad = 0;
  for (int dev = 0; dev < 8; ++dev) {
    c.device = dev & 1, d.device = (dev >> 1) & 1, s.device = (dev >> 2) & 1;
    kernels = copies = 0;
    fcopy(&c, &d, &s);
    const bool one = c.device == d.device && c.device == s.device;
    if (one ? kernels != 1 || copies : kernels || copies != 2) {
      std::printf("context %d, from %d to %d: %d kernels, %d copies\n", c.device, s.device, d.device, kernels, copies);
      ++bad;
    }
  }
  return bad;
}
'''


def test_copy_between_devices(tmp_path):
    src, obj, exe = tmp_path / 'fcopy.hip', tmp_path / 'fcopy.o', tmp_path / 'fcopy'
    src.write_text(DRIVER.replace('CAPI_SOURCE', os.path.join(build.CSRC, 'capi.hip')))
    subprocess.run([build.HIPCC, '--cuda-host-only', '-std=c++17', '-O1', '-fPIC',
                    '-I' + os.path.join(build.ROOT, 'include'), '-I' + build.CSRC, '-c', str(src), '-o', str(obj)],
                   check=True, timeout=300)
    subprocess.run(['g++', str(obj), '-Wl,--unresolved-symbols=ignore-all', '-o', str(exe)], check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
