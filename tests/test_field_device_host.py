"""A field made while another device than its context's is current (a process with
contexts on several devices): its memory lies on the current device, and is kept for
that device's fields.  On the CPU, with the runtime's calls replaced."""
import os
import subprocess

from mlegs_amd import build

DRIVER = r'''
#include "CAPI_SOURCE"
#include <cstdio>
#include <cstdlib>
static int got = -1, put = -1;
extern "C" {
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *,
                           int *) {}
void __hipUnregisterFatBinary(void **) {}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
  *s = hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) { return *d = 3, hipSuccess; }
}
namespace mlx {
void *field_mem_get(int device, size_t n) { return got = device, std::malloc(n); }
void field_mem_put(int device, void *p, size_t) { put = device, std::free(p); }
void k_zero_field(mlx_ctx *, double2 *, double *) {}
}
int main() {
  mlx_ctx c;
  c.nelem = 10;
  c.device = 1;
  mlx_field *f = field_new(&c);
  const int at = f->device;
  field_free(f);
  std::printf("taken from device %d, the field's %d, given to %d\n", got, at, put);
  return !(got == 3 && at == 3 && put == 3);
}
'''


def test_device_of_a_field(tmp_path):
    src, obj, exe = tmp_path / 'fdev.hip', tmp_path / 'fdev.o', tmp_path / 'fdev'
    src.write_text(DRIVER.replace('CAPI_SOURCE', os.path.join(build.CSRC, 'capi.hip')))
    subprocess.run([build.HIPCC, '--cuda-host-only', '-std=c++17', '-O1', '-fPIC',
                    '-I' + os.path.join(build.ROOT, 'include'), '-I' + build.CSRC, '-c', str(src), '-o', str(obj)],
                   check=True, timeout=300)
    subprocess.run(['g++', str(obj), '-Wl,--unresolved-symbols=ignore-all', '-o', str(exe)], check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
