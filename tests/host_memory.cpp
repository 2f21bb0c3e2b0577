// Device buffers, their pool and the host copies of pssa_amd/csrc/common.h on
// the CPU: the runtime's memory calls are replaced by a heap of a fixed size.
// Prints one line per check that fails; the exit status is their number.
#include "../pssa_amd/csrc/common.h"

#include <cstdlib>

namespace {
size_t g_capacity, g_used, g_copies;
std::map<void*, size_t> g_blocks;
int g_failed = 0;

void check(bool ok, const char* what) {
  if (ok) return;
  std::printf("failed: %s\n", what);
  ++g_failed;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (g_used + n > g_capacity) return hipErrorOutOfMemory;
  *p = std::malloc(64);
  g_blocks[*p] = n;
  g_used += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  const auto it = g_blocks.find(p);
  if (it == g_blocks.end()) return hipErrorInvalidValue;
  g_used -= it->second;
  g_blocks.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::malloc(n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
  ++g_copies;
  std::memcpy(dst, src, n);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t*, const void*) { return hipErrorInvalidValue; }
}

using pssa::DevBuf;
using pssa::DevPool;

// Every allocation of the library, pooled or not and of whichever context,
// finds the memory that pools hold.
static void pool_gives_way() {
  constexpr size_t MB = (size_t)1 << 20;
  g_capacity = 200 * MB;
  DevPool a, b;
  {
    DevBuf x, y;
    check(x.alloc(80 * MB, &a).ok() && y.alloc(60 * MB, &b).ok(), "first allocations");
  }
  check(g_used == 140 * MB, "blocks are held for the next call");
  {
    DevBuf again;
    check(again.alloc(70 * MB, &a).ok() && g_used == 140 * MB && again.bytes == 80 * MB, "a held block is handed out");
    DevBuf model;  // not pooled: 60 MB free, 60 more held by the other context
    check(model.alloc(100 * MB).ok(), "an unpooled buffer takes the place of held blocks");
  }
  check(g_used == 80 * MB, "the unpooled buffer is freed, the pooled one held");
  void* p = nullptr;
  check(pssa::device_malloc(&p, 190 * MB) == hipSuccess && p, "a plain allocation takes the place of held blocks");
  DevBuf z;
  check(!z.alloc(20 * MB, &a).ok() && z.p == nullptr && z.pool == nullptr, "no memory is an error");
  void* q = &z;
  check(pssa::device_malloc(&q, 20 * MB) == hipErrorOutOfMemory && !q, "no memory, nothing held");
  (void)hipFree(p);
  check(z.alloc(20 * MB, &a).ok(), "and memory again");
}

int main() {
  pool_gives_way();
  check(g_used == 0, "pools and buffers free everything");
  return g_failed;
}
