// Device buffers, their pool and the host copies of pssa_amd/csrc/common.h on
// the CPU: the runtime's memory calls are replaced by a heap of a fixed size
// and a stream that runs the copies of pinned memory only when it is waited for.
// Prints one line per check that fails; the exit status is their number.
#include "../pssa_amd/csrc/common.h"

#include <cstdlib>

namespace {
size_t g_capacity, g_used;
std::map<void*, size_t> g_blocks;
std::map<const char*, size_t> g_pinned;    // of hipHostMalloc
std::vector<std::tuple<char*, const char*, size_t>> g_queue, g_direct;
const void* g_device = nullptr;            // a device array
int g_failed = 0;

bool pinned(const void* q) {
  const char* p = static_cast<const char*>(q);
  auto it = g_pinned.upper_bound(p);
  return it != g_pinned.begin() && p < std::prev(it)->first + std::prev(it)->second;
}
void run_queue() {
  for (auto& [dst, src, n] : g_queue) std::memcpy(dst, src, n);
  g_queue.clear();
}

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
  g_pinned[static_cast<char*>(*p)] = n;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  g_pinned.erase(static_cast<char*>(p));
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
  g_queue.emplace_back(static_cast<char*>(dst), static_cast<const char*>(src), n);
  if (pinned(dst) || pinned(src)) return hipSuccess;
  g_direct.push_back(g_queue.back());
  run_queue();
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  run_queue();
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* at, const void* p) {
  std::memset(at, 0, sizeof(*at));
  at->type = p == g_device ? hipMemoryTypeDevice : pinned(p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return hipSuccess;
}
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

// Arrays of all sizes around the slots up and down, several uploads before a
// wait; and memory the runtime knows is left to it.
static void copies() {
  constexpr size_t K = 1024, S = pssa::HostStage::kSlot, M = pssa::HostStage::kMin;
  pssa::HostStage st;
  check(st.init().ok(), "slots");
  const size_t sizes[] = {1, M - 1, M, M + 1, 700 * K + 3, S - 1, S, S + 1, 3 * S, 5 * S + 77};
  for (size_t n : sizes) {
    std::vector<std::vector<unsigned char>> dst(9, std::vector<unsigned char>(n));
    for (size_t r = 0; r < dst.size(); ++r) {
      std::vector<unsigned char> src(n);
      for (size_t i = 0; i < n; ++i) src[i] = (unsigned char)(i * 7 + i / 251 + r);
      check(st.to_device(dst[r].data(), src.data(), n, nullptr).ok(), "to_device");
      std::fill(src.begin(), src.end(), 0xEE);  // reused at once
    }
    std::vector<unsigned char> back(n);
    check(st.to_host(back.data(), dst[8].data(), n, nullptr).ok() && st.wait(nullptr).ok(), "to_host");
    bool same = back == dst[8];
    for (size_t r = 0; r < dst.size(); ++r)
      for (size_t i = 0; i < n; ++i) same &= dst[r][i] == (unsigned char)(i * 7 + i / 251 + r);
    check(same, ("copies of " + std::to_string(n) + " bytes").c_str());
  }
  for (size_t n : sizes) {
    std::vector<char> a(n, 1), b(n, 2);
    g_device = a.data();
    g_direct.clear();
    check(st.to_device(b.data(), a.data(), n, nullptr).ok() && st.to_host(a.data(), b.data(), n, nullptr).ok() &&
              st.wait(nullptr).ok(),
          "copies");
    check(g_direct.size() == 2 && std::get<1>(g_direct[0]) == a.data() && std::get<2>(g_direct[0]) == n &&
              std::get<0>(g_direct[1]) == a.data() && std::get<2>(g_direct[1]) == n,
          ("a device array of " + std::to_string(n) + " bytes is copied by the runtime alone").c_str());
  }
}

int main() {
  pool_gives_way();
  check(g_used == 0, "pools and buffers free everything");
  copies();
  return g_failed;
}
