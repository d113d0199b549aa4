// pool.cpp -- large device blocks kept between objects.
//
// A program that makes a diagram per time step allocates and frees the same
// large arrays each time, and the runtime maps and unmaps them: a hipMalloc
// and hipFree pair costs 1.3 us up to 1.5 MiB (the runtime suballocates
// those), 26 us from 2 MiB and 260 us from 128 MiB on.  Blocks of kPoolMin
// and more are therefore kept when they are freed and handed out again.  A
// diagram made, computed and destroyed: 22.6 -> 19.0 ms at 1M uniform points,
// 6.0 -> 4.9 ms at 256k of a perturbed lattice.
//
// What an allocation and a free mean to the caller stays what it was.  Every
// block carries a token, a small allocation of its own, made when the block
// is handed out and freed when it comes back: where the runtime refuses an
// allocation (a stream of the process is being captured) the token is refused
// and the block with it, and freeing the token waits for all work on the
// device, as hipFree does, so nothing still reads or writes a block when the
// next object gets it, whichever stream, thread or context that one is on.
//
// Bounded: at most 1/64 of the device's memory is kept, oldest blocks given
// back first; a block is handed out for requests of at least 8/9 of it; all
// of it is given back when a device allocation of any size finds no memory
// (and that is tried once more), and when the last context on the device is
// destroyed.
#include <hip/hip_runtime.h>

#include <list>
#include <mutex>
#include <vector>

#include "runtime.h"

namespace tess {

namespace {

constexpr int kMaxDevices = 64;
constexpr size_t kTokenBytes = 64;

struct KeptBlock {
  void* p;
  size_t bytes;
};

struct DevicePool {
  std::mutex mu;
  std::list<KeptBlock> kept;  // oldest first
  size_t bytes = 0, limit = 0;
  int contexts = 0;
};

// never destroyed: objects may be freed while the process ends
DevicePool* pools() {
  static DevicePool* p = new DevicePool[kMaxDevices];
  return p;
}

DevicePool* pool_of(int device) { return device >= 0 && device < kMaxDevices ? pools() + device : nullptr; }

void give_back_all(DevicePool& P) {
  std::list<KeptBlock> out;
  {
    std::lock_guard<std::mutex> g(P.mu);
    out.swap(P.kept);
    P.bytes = 0;
  }
  for (const KeptBlock& b : out) (void)hipFree(b.p);
}

DevicePool* current_pool(int* device) {
  if (hipGetDevice(device) != hipSuccess) *device = -1;
  return pool_of(*device);
}

}  // namespace

hipError_t device_alloc(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  int device = -1;
  DevicePool* P = e == hipErrorOutOfMemory ? current_pool(&device) : nullptr;
  if (P) {
    (void)hipGetLastError();
    give_back_all(*P);
    e = hipMalloc(p, bytes);
  }
  if (e != hipSuccess) *p = nullptr;
  return e;
}

void pool_context_add(int device) {
  DevicePool* P = pool_of(device);
  if (!P) return;
  std::lock_guard<std::mutex> g(P->mu);
  size_t total = 0;
  if (!P->limit && hipDeviceTotalMem(&total, device) == hipSuccess) P->limit = total / 64;
  ++P->contexts;
}

void pool_context_remove(int device) {
  DevicePool* P = pool_of(device);
  if (!P) return;
  {
    std::lock_guard<std::mutex> g(P->mu);
    if (--P->contexts > 0) return;
  }
  give_back_all(*P);
}

hipError_t pool_alloc(size_t bytes, PoolBlock* out) {
  *out = PoolBlock{};
  int device = -1;
  DevicePool* P = current_pool(&device);
  hipError_t e = device_alloc(&out->token, kTokenBytes);
  if (e != hipSuccess) return e;
  if (P) {
    std::lock_guard<std::mutex> g(P->mu);
    auto best = P->kept.end();
    for (auto it = P->kept.begin(); it != P->kept.end(); ++it)
      if (it->bytes >= bytes && it->bytes - bytes <= bytes / 8 &&
          (best == P->kept.end() || it->bytes < best->bytes))
        best = it;
    if (best != P->kept.end()) {
      out->p = best->p;
      out->bytes = best->bytes;
      P->bytes -= best->bytes;
      P->kept.erase(best);
    }
  }
  if (!out->p) {
    e = device_alloc(&out->p, bytes);
    if (e != hipSuccess) {
      (void)hipFree(out->token);
      *out = PoolBlock{};
      return e;
    }
    out->bytes = bytes;
  }
  out->device = device;
  return hipSuccess;
}

void pool_free(const PoolBlock& b) {
  if (!b.p) return;
  DevicePool* P = pool_of(b.device);
  // a token that cannot be freed has not waited: the block is not kept
  if (hipFree(b.token) != hipSuccess || !P) {
    (void)hipFree(b.p);
    return;
  }
  std::list<KeptBlock> out;
  bool keep;
  {
    std::lock_guard<std::mutex> g(P->mu);
    keep = P->contexts > 0 && b.bytes <= P->limit;
    if (keep) {
      while (P->bytes + b.bytes > P->limit && !P->kept.empty()) {
        P->bytes -= P->kept.front().bytes;
        out.splice(out.end(), P->kept, P->kept.begin());
      }
      try {
        P->kept.push_back({b.p, b.bytes});
        P->bytes += b.bytes;
      } catch (...) {
        keep = false;
      }
    }
  }
  for (const KeptBlock& o : out) (void)hipFree(o.p);
  if (!keep) (void)hipFree(b.p);
}

}  // namespace tess
