// Device memory of fields, kept between one field's end and the next one's
// start.
//
// hipFree waits for the whole device and unmaps, hipMalloc maps: about 110 and
// 20 us for a field, with the GPU idle meanwhile.  Code that makes copies as it
// goes paid that for each: a gradient of twelve steps at 128 x 64 x 64 frees
// 120 blocks, 13 of its 24 ms.
//
// A freed block waits in `limbo` until a hipFree has passed, whose implicit wait
// for the device covers the work of every stream that was issued before the
// block was given up, the caller's own streams included; only then is it handed
// out again.  32 blocks in limbo are enough for one such hipFree (of the
// smallest of them).  A hipFree that fails (it is refused while any stream of the
// process records a graph) has waited for nothing: its block and limbo stay as
// they are until a later one succeeds.  What is kept is bounded per device
// (kMaxBytes, kMaxBlocks; a block over kMaxBlock is freed at once; at a bound the
// largest ready block of another size goes instead, so that a size no longer in
// use does not hold the place), and is returned when an allocation of this
// library finds no memory, when the last kit with fields of a block's size ends,
// and when the device's last context does.  (Returning everything with any
// context costs the first pass on the next kit of the same size its allocations:
// 17.4 against 13.4 ms of a vortex step at 256^3.)  Blocks are matched by size
// alone, under a mutex: no owner, stream or address plays a part.
#include <mutex>

#include "mlx_internal.h"

namespace {

constexpr size_t kMaxBytes = (size_t)2 << 30;
constexpr size_t kMaxBlock = kMaxBytes / 8;
constexpr size_t kMaxBlocks = 256, kLimbo = 32;

struct Block {
  void *p;
  size_t bytes;
};
struct Pool {
  std::vector<Block> limbo, ready;
  size_t bytes = 0;  // of both
  int contexts = 0;
  std::map<size_t, int> kits;  // by the size of their fields

  // whether b was freed, which is also whether the device has been waited for
  bool drop(Block b) {
    if (hipFree(b.p) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    bytes -= b.bytes;
    return true;
  }
  // frees the blocks of one size (0: all)
  void release(size_t size = 0) {
    for (auto *v : {&limbo, &ready}) {
      size_t left = 0;
      for (size_t i = 0; i < v->size(); ++i)
        if ((size && (*v)[i].bytes != size) || !drop((*v)[i])) (*v)[left++] = (*v)[i];
      v->resize(left);
    }
  }
};

std::mutex g_mutex;
std::map<int, Pool> &pools() {
  static auto *p = new std::map<int, Pool>;  // outlives every static destructor
  return *p;
}

}  // namespace

namespace mlx {

void *field_mem_get(int device, size_t bytes) {
  {
    std::lock_guard<std::mutex> lock(g_mutex);
    Pool &q = pools()[device];
    for (size_t i = q.ready.size(); i-- > 0;)
      if (q.ready[i].bytes == bytes) {
        void *p = q.ready[i].p;
        q.ready[i] = q.ready.back();
        q.ready.pop_back();
        q.bytes -= bytes;
        return p;
      }
  }
  void *p = nullptr;
  return dev_malloc(&p, bytes) == hipSuccess ? p : nullptr;
}

void field_mem_put(int device, void *p, size_t bytes) {
  if (!p) return;
  std::lock_guard<std::mutex> lock(g_mutex);
  Pool &q = pools()[device];
  q.limbo.push_back({p, bytes});
  q.bytes += bytes;
  if (q.contexts <= 0) {
    q.release();
    return;
  }
  // the block to free: this one where it is not to be kept, another size's in
  // its place where that is enough, else the smallest of a full limbo
  const size_t over_bytes = q.bytes > kMaxBytes ? q.bytes - kMaxBytes : 0;
  const bool over = over_bytes > 0 || q.limbo.size() + q.ready.size() > kMaxBlocks;
  std::vector<Block> *from = &q.limbo;
  size_t out = q.limbo.size() - 1;
  if (bytes <= kMaxBlock && over) {
    size_t most = 0;
    for (size_t i = 0; i < q.ready.size(); ++i)
      if (q.ready[i].bytes != bytes && q.ready[i].bytes >= over_bytes && q.ready[i].bytes > most)
        from = &q.ready, most = q.ready[out = i].bytes;
  } else if (bytes <= kMaxBlock) {
    if (q.limbo.size() < kLimbo) return;
    for (size_t i = 0; i < q.limbo.size(); ++i)
      if (q.limbo[i].bytes < q.limbo[out].bytes) out = i;
  }
  if (!q.drop((*from)[out])) return;
  from->erase(from->begin() + out);
  // the hipFree has waited for all work on the device
  q.ready.insert(q.ready.end(), q.limbo.begin(), q.limbo.end());
  q.limbo.clear();
}

bool field_mem_release(int device) {
  std::lock_guard<std::mutex> lock(g_mutex);
  Pool &q = pools()[device];
  const size_t held = q.bytes;
  q.release();
  return q.bytes < held;
}

void field_mem_contexts(int device, int d) {
  std::lock_guard<std::mutex> lock(g_mutex);
  Pool &q = pools()[device];
  q.contexts += d;
  if (q.contexts <= 0) q.release();
}

void field_mem_kits(int device, size_t bytes, int d) {
  std::lock_guard<std::mutex> lock(g_mutex);
  Pool &q = pools()[device];
  if ((q.kits[bytes] += d) > 0) return;
  q.kits.erase(bytes);
  q.release(bytes);
}

}  // namespace mlx
