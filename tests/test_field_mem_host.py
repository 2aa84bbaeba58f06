"""The bookkeeping of kept field memory (csrc/field_mem.hip) on the CPU, with
hipMalloc and hipFree replaced: a block that was given up is handed out again
only after a hipFree that succeeded, which is what waits for the device; and
what is kept is given back with the last kit of its size and makes room for other
sizes."""
import os
import subprocess

import pytest

from mlegs_amd import build

DRIVER = r'''
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>
#include <vector>

#include <hip/hip_runtime.h>

static std::set<void *> live;  // allocated, not freed
static bool refuse = false;    // hipFree fails, as while a stream records a graph
static int frees = 0;
extern "C" hipError_t hipMalloc(void **p, size_t n) {
  live.insert(*p = std::malloc(n));
  return hipSuccess;
}
extern "C" hipError_t hipFree(void *p) {
  if (refuse) return hipErrorStreamCaptureUnsupported;
  if (!live.erase(p)) std::abort();
  std::free(p);
  ++frees;
  return hipSuccess;
}
extern "C" hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
extern "C" hipError_t hipGetLastError() { return hipSuccess; }

namespace mlx {
void *field_mem_get(int device, size_t bytes);
void field_mem_put(int device, void *p, size_t bytes);
bool field_mem_release(int device);
void field_mem_contexts(int device, int d);
void field_mem_kits(int device, size_t bytes, int d);
}
using namespace mlx;

#define CHECK(x)                                          \
  do {                                                    \
    if (!(x)) return std::printf("line %d: %s\n", __LINE__, #x), 1; \
  } while (0)

static std::vector<void *> some(int n, size_t bytes) {
  std::vector<void *> v;
  for (int i = 0; i < n; ++i) v.push_back(field_mem_get(0, bytes));
  return v;
}
// whether any of v is among what the next n requests get
static bool again(const std::vector<void *> &v, int n, size_t bytes) {
  bool hit = false;
  std::vector<void *> w = some(n, bytes);
  for (void *p : v)
    for (void *q : w) hit |= p == q;
  return hit;
}

// the limbo's hipFree is refused: nothing given up may be handed out, nothing is lost
static int refused_limbo() {
  field_mem_contexts(0, 1);
  std::vector<void *> v = some(100, 64);
  const size_t n = live.size();
  refuse = true;
  for (void *p : v) field_mem_put(0, p, 64);
  CHECK(live.size() == n);
  CHECK(!again(v, 100, 64));
  refuse = false;
  void *one = field_mem_get(0, 64);
  field_mem_put(0, one, 64);  // tried again: the wait has now taken place
  CHECK(frees == 1);
  CHECK(again(v, 60, 64));
  return 0;
}

// a block too large to be kept whose hipFree is refused stays until a later one succeeds
static int refused_large() {
  const size_t big = (size_t)300 << 20;
  field_mem_contexts(0, 1);
  std::vector<void *> v = some(5, 64);
  void *b = field_mem_get(0, big);
  for (void *p : v) field_mem_put(0, p, 64);
  refuse = true;
  field_mem_put(0, b, big);
  CHECK(!again(v, 5, 64));
  CHECK(live.count(b));
  refuse = false;
  for (void *p : some(40, 64)) field_mem_put(0, p, 64);
  field_mem_release(0);
  CHECK(!live.count(b));
  return 0;
}

// a release that is refused gives nothing back and loses nothing
static int refused_release() {
  field_mem_contexts(0, 1);
  for (void *p : some(5, 64)) field_mem_put(0, p, 64);
  refuse = true;
  CHECK(!field_mem_release(0));
  field_mem_contexts(0, -1);
  CHECK(live.size() == 5);
  refuse = false;
  CHECK(field_mem_release(0));
  CHECK(live.empty());
  CHECK(!field_mem_release(0));
  return 0;
}

// the last kit with fields of a size gives that size back, also while other contexts of the device live
static int kit_end() {
  for (int i = 0; i < 3; ++i) field_mem_contexts(0, 1);
  field_mem_kits(0, 4096, 1);
  field_mem_kits(0, 4096, 1);
  field_mem_kits(0, 8192, 1);
  std::vector<void *> a = some(40, 4096), b = some(40, 8192);
  for (int i = 0; i < 40; ++i) field_mem_put(0, a[i], 4096), field_mem_put(0, b[i], 8192);
  const size_t all = live.size();
  field_mem_kits(0, 4096, -1);
  field_mem_contexts(0, -1);
  CHECK(live.size() == all);  // the other kit's fields may still take them
  field_mem_kits(0, 4096, -1);
  field_mem_contexts(0, -1);
  for (void *p : a) CHECK(!live.count(p));
  CHECK(!live.empty());
  field_mem_kits(0, 8192, -1);
  CHECK(live.empty());
  return 0;
}

// kept blocks of a size that is no longer asked for make room for the size that is
static int other_size() {
  const size_t old = (size_t)64 << 20;  // 32 of them are all that is kept
  field_mem_contexts(0, 1);
  for (void *p : some(64, old)) field_mem_put(0, p, old);
  for (int round = 0; round < 40; ++round)
    for (void *p : some(20, 1 << 20)) field_mem_put(0, p, 1 << 20);
  const int before = frees;
  for (int round = 0; round < 40; ++round)
    for (void *p : some(20, 1 << 20)) field_mem_put(0, p, 1 << 20);
  CHECK(frees - before <= 40);  // 800 when each goes straight to hipFree
  return 0;
}

int main(int, char **argv) {
  const struct { const char *name; int (*fn)(); } all[] = {
      {"refused_limbo", refused_limbo}, {"refused_large", refused_large}, {"refused_release", refused_release},
      {"kit_end", kit_end}, {"other_size", other_size}};
  for (auto &t : all)
    if (!std::strcmp(argv[1], t.name)) return t.fn();
  return 2;
}
'''


@pytest.fixture(scope='module')
def driver(tmp_path_factory):
    d = tmp_path_factory.mktemp('field_mem')
    src, exe = d / 'driver.hip', d / 'driver'
    src.write_text(DRIVER)
    host = [build.HIPCC, '--cuda-host-only', '-std=c++17', '-O1', '-fPIC', '-I' + os.path.join(build.ROOT, 'include')]
    objs = []
    for s in (str(src), os.path.join(build.CSRC, 'field_mem.hip')):
        objs.append(str(d / (os.path.basename(s) + '.o')))
        subprocess.run(host + ['-c', s, '-o', objs[-1]], check=True, timeout=300)
    subprocess.run(['g++'] + objs + ['-lpthread', '-o', str(exe)], check=True, timeout=120)
    return str(exe)


@pytest.mark.parametrize('case', ['refused_limbo', 'refused_large', 'refused_release', 'kit_end', 'other_size'])
def test_field_mem(driver, case):
    r = subprocess.run([driver, case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
