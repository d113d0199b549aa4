// Host check of the kept device blocks (csrc/pool.cpp, DevBuf): the runtime's
// allocator is replaced by one over a counted amount of memory.
#include <cstdio>
#include <cstdlib>
#include <map>

#include "../the-tessellator_amd/csrc/runtime.h"

namespace {
size_t room = 0;  // bytes left
bool captured = false;
std::map<void*, size_t> live;
int refused = 0;
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
  if (captured) return hipErrorStreamCaptureUnsupported;
  if (bytes > room) {
    ++refused;
    return hipErrorOutOfMemory;
  }
  room -= bytes;
  *p = std::malloc(1);
  live[*p] = bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (!p) return hipSuccess;
  if (!live.count(p)) std::abort();
  room += live[p];
  live.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipDeviceTotalMem(size_t* b, hipDevice_t) { return *b = size_t(64) << 23, hipSuccess; }  // keeps 8 MiB
}

#define CHECK(c) \
  if (!(c)) return std::printf("line %d: %s\n", __LINE__, #c), 1

int main() {
  using namespace tess;
  constexpr size_t kBlock = size_t(3) << 20;
  auto kept = [] {  // 3 MiB kept, nothing left beside it
    room = kBlock + 64;
    DevBuf<char> a;
    if (a.alloc(kBlock) != hipSuccess) std::abort();
    a.reset();
    room = 0;
    return live.size();
  };
  pool_context_add(0);
  // an allocation that the runtime suballocates
  CHECK(kept() == 1);
  {
    DevBuf<char> b;
    CHECK(b.alloc(1000) == hipSuccess && b.p && live.size() == 1);
  }
  // a large one's token, for a block that the kept one does not serve
  CHECK(kept() == 1);
  {
    DevBuf<char> b;
    CHECK(b.alloc(kBlock - (size_t(1) << 19)) == hipSuccess && live.size() == 2);
  }
  CHECK(live.size() == 1);
  pool_context_remove(0);
  CHECK(live.empty());
  pool_context_add(0);
  // a large one itself
  CHECK(kept() == 1);
  room = 64;
  {
    DevBuf<char> b;
    CHECK(b.alloc(kBlock - (size_t(1) << 19)) == hipSuccess && live.size() == 2);
  }
  pool_context_remove(0);
  CHECK(live.empty());
  pool_context_add(0);
  // nothing kept, nothing left: refused, nothing lost
  room = 100;
  {
    DevBuf<char> b;
    CHECK(b.alloc(1000) == hipErrorOutOfMemory && !b.p && b.n == 0);
    CHECK(b.alloc(kBlock) == hipErrorOutOfMemory && !b.p && b.n == 0);
    CHECK(b.alloc(100) == hipSuccess);
  }
  CHECK(live.empty() && room == 100);
  // an error that is not want of memory gives nothing back
  CHECK(kept() == 1);
  captured = true;
  refused = 0;
  {
    DevBuf<char> b;
    CHECK(b.alloc(1000) == hipErrorStreamCaptureUnsupported && b.alloc(kBlock) == hipErrorStreamCaptureUnsupported);
  }
  captured = false;
  CHECK(live.size() == 1 && refused == 0);
  pool_context_remove(0);
  CHECK(live.empty());
  std::printf("kept blocks: as stated\n");
  return 0;
}
