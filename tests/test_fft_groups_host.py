"""The grouping of an FFT plan's passes (csrc/fft.hip, groups_of) on the CPU: for
every length the kernels take, and the radices in any order, the groups are ones
that a kernel exists for, cover the length, and fit the workgroup's LDS."""
import os
import subprocess

from mlegs_amd import build

DRIVER = r'''
#include "FFT_SOURCE"
#include <algorithm>
#include <cstdio>
#include <random>
extern "C" {  // no device code in this program
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *,
                           int *) {}
void __hipUnregisterFatBinary(void **) {}
}
int main() {
  const int built[] = {0x44, 0x42, 0x43, 0x41, 0x23, 0x25, 0x21, 0x33, 0x35, 0x31, 0x51, 0x11};
  std::mt19937 rng(1);
  int bad = 0, plans = 0;
  for (int n = 1; n <= 512; ++n)
    for (int t = 0; t < 200; ++t) {
      FftPlan pl{};
      pl.n = n;
      int r = n;
      for (int f : {4, 2, 3, 5})  // the library's own order at t = 0
        while (r % f == 0 && !(f == 4 && t % 2 && rng() % 2)) pl.radix[pl.npass++] = f, r /= f;
      if (r != 1) break;
      if (t) std::shuffle(pl.radix, pl.radix + pl.npass, rng);
      ++plans;
      for (int nwg : {1, 64, 4096}) {
        FftGroups g;
        try {
          g = groups_of(pl, 264, nwg);
        } catch (const MlxError &) {
          bad += t == 0;  // refused only where the library does not order them so
          continue;
        }
        int ns = 1;
        bool ok = g.n == n && g.til >= 2 && ((size_t)n << g.til) * 32 <= 65536;
        for (int i = 0; i < g.ng; ++i) {
          ok = ok && g.ns[i] == ns && std::count(std::begin(built), std::end(built), g.type[i]);
          ns *= (g.type[i] / 16) * (g.type[i] % 16);
        }
        if (!ok || ns != n) {
          if (++bad < 5) std::printf("n %d order %d: %d groups, first %x\n", n, t, g.ng, g.type[0]);
        }
      }
    }
  std::printf("%d plans, %d bad\n", plans, bad);
  return bad != 0 || plans < 10000;
}
'''


def test_groups(tmp_path):
    src, obj, exe = tmp_path / 'groups.hip', tmp_path / 'groups.o', tmp_path / 'groups'
    src.write_text(DRIVER.replace('FFT_SOURCE', os.path.join(build.CSRC, 'fft.hip')))
    subprocess.run([build.HIPCC, '--cuda-host-only', '-std=c++17', '-O1', '-fPIC',
                    '-I' + os.path.join(build.ROOT, 'include'), '-I' + build.CSRC, '-c', str(src), '-o', str(obj)],
                   check=True, timeout=300)
    # the HIP runtime is not called
    subprocess.run(['g++', str(obj), '-Wl,--unresolved-symbols=ignore-all', '-o', str(exe)], check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
