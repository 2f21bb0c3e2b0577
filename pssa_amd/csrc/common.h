// Shared host/device helpers for libpssa_hip (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/pssa_hip.h"

namespace pssa {

// Error carrier used inside the library; converted to (code, message) at the
// C boundary.
struct Status {
  int code = PSSA_HIP_OK;
  std::string msg;
  bool ok() const { return code == PSSA_HIP_OK; }
  static Status Ok() { return {}; }
  static Status Invalid(const std::string& m) { return {PSSA_HIP_EINVAL, m}; }
  static Status Device(const std::string& m) { return {PSSA_HIP_EDEVICE, m}; }
  static Status NoMem(const std::string& m) { return {PSSA_HIP_ENOMEM, m}; }
  static Status NoDev(const std::string& m) { return {PSSA_HIP_ENODEV, m}; }
};

inline int finish(const Status& s, char* err, size_t err_len) {
  if (err && err_len) {
    if (s.ok()) {
      err[0] = 0;
    } else {
      std::snprintf(err, err_len, "%s", s.msg.c_str());
    }
  }
  return s.code;
}

#define PSSA_RETURN_IF(st) \
  do {                     \
    Status _s = (st);      \
    if (!_s.ok()) return _s; \
  } while (0)

#define PSSA_HIP_TRY(expr)                                                              \
  do {                                                                                  \
    hipError_t _e = (expr);                                                             \
    if (_e != hipSuccess)                                                               \
      return Status::Device(std::string(#expr) + ": " + hipGetErrorString(_e));          \
  } while (0)

// Launch check: a failed launch configuration is reported at the call site.
#define PSSA_LAUNCH_CHECK(name)                                                         \
  do {                                                                                  \
    hipError_t _e = hipGetLastError();                                                  \
    if (_e != hipSuccess)                                                               \
      return Status::Device(std::string("launch ") + (name) + ": " + hipGetErrorString(_e)); \
  } while (0)

inline bool mul_ok(size_t a, size_t b, size_t* out) {
  if (a != 0 && b > SIZE_MAX / a) return false;
  *out = a * b;
  return true;
}
inline Status checked_count(std::initializer_list<size_t> dims, size_t* out, const char* what) {
  size_t n = 1;
  for (size_t d : dims)
    if (!mul_ok(n, d, &n)) return Status::Invalid(std::string(what) + ": element count overflow");
  if (n > ((size_t)1 << 40)) return Status::Invalid(std::string(what) + ": too large");
  *out = n;
  return Status::Ok();
}

// Device blocks kept between calls for the temporaries of the host-array
// entry points (a call takes up to fifteen; a hipMalloc / hipFree pair of 6 MB
// costs 23 us, of up to 1 MiB 1.3).  Blocks are handed out again on the
// context's one stream, so a block's next user runs after its last; at most
// kPoolBytes are held, the rest is freed at once, and all of it with the
// context or when an allocation of any context finds no memory (device_malloc).
class DevPool {
 public:
  static constexpr size_t kPoolBytes = (size_t)256 << 20;
  DevPool() {
    std::lock_guard<std::mutex> g(pools().mu);
    next_ = pools().first;
    pools().first = this;
  }
  ~DevPool() {
    {
      std::lock_guard<std::mutex> g(pools().mu);
      DevPool** at = &pools().first;
      while (*at != this) at = &(*at)->next_;
      *at = next_;
    }
    clear();
  }
  DevPool(const DevPool&) = delete;
  DevPool& operator=(const DevPool&) = delete;
  // Frees what every pool of the process holds; false if that was nothing.
  static bool clear_all() {
    std::lock_guard<std::mutex> g(pools().mu);
    bool any = false;
    for (DevPool* p = pools().first; p; p = p->next_) any |= p->clear();
    return any;
  }
  // A held block of at least `n` bytes and not much more, or null.
  void* take(size_t n, size_t* bytes) {
    std::lock_guard<std::mutex> g(mu_);
    const auto it = free_.lower_bound(n);
    if (it == free_.end() || it->first > 2 * n + 4096) return nullptr;
    void* p = it->second;
    *bytes = it->first;
    held_ -= it->first;
    free_.erase(it);
    return p;
  }
  void put(void* p, size_t bytes) {
    {
      std::lock_guard<std::mutex> g(mu_);
      if (held_ + bytes <= kPoolBytes) {
        try {
          free_.emplace(bytes, p);
          held_ += bytes;
          return;
        } catch (...) {  // no host memory to hold it: freed (destructors call this)
        }
      }
    }
    (void)hipFree(p);
  }
  bool clear() {
    std::lock_guard<std::mutex> g(mu_);
    const bool any = !free_.empty();
    for (auto& f : free_) (void)hipFree(f.second);
    free_.clear();
    held_ = 0;
    return any;
  }

 private:
  struct All {
    std::mutex mu;
    DevPool* first = nullptr;
  };
  static All& pools() {
    static All* all = new All;  // outlives every context
    return *all;
  }
  DevPool* next_ = nullptr;
  std::mutex mu_;
  std::multimap<size_t, void*> free_;
  size_t held_ = 0;
};

// hipMalloc; with no memory left, again without the blocks that pools hold.
inline hipError_t device_malloc(void** p, size_t n) {
  hipError_t e = hipMalloc(p, n);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    if (DevPool::clear_all()) e = hipMalloc(p, n);
    if (e != hipSuccess) (void)hipGetLastError();
  }
  if (e != hipSuccess) *p = nullptr;
  return e;
}

// Device buffer owned by RAII (returned to `pool` when it came from one).
struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
  DevPool* pool = nullptr;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  DevBuf(DevBuf&& o) noexcept : p(o.p), bytes(o.bytes), pool(o.pool) {
    o.p = nullptr;
    o.bytes = 0;
  }
  DevBuf& operator=(DevBuf&& o) noexcept {
    if (this != &o) {
      release();
      p = o.p;
      bytes = o.bytes;
      pool = o.pool;
      o.p = nullptr;
      o.bytes = 0;
    }
    return *this;
  }
  ~DevBuf() { release(); }
  void release() {
    if (p && pool)
      pool->put(p, bytes);
    else if (p)
      (void)hipFree(p);
    p = nullptr;
    bytes = 0;
    pool = nullptr;
  }
  Status alloc(size_t n, DevPool* from = nullptr) {
    release();
    n = (n + 255) & ~(size_t)255;  // whole 256-byte granules: fills may round up to a vector
    if (n == 0) n = 256;
    if (from && (p = from->take(n, &bytes))) {
      pool = from;
      return Status::Ok();
    }
    const hipError_t e = device_malloc(&p, n);
    if (e != hipSuccess) return Status::NoMem("hipMalloc(" + std::to_string(n) + "): " + hipGetErrorString(e));
    bytes = n;
    pool = from;
    return Status::Ok();
  }
  template <class T>
  T* as() const {
    return static_cast<T*>(p);
  }
};

// Copies between host arrays and the device.  The runtime's copies of
// pageable arrays cost 105 us for 256 KiB either way and 330-370 us down for 6
// MB on the machine measured; a pinned transfer and a memcpy 13 + 9 us, and
// with the host's copy of one piece beside the transfer of the next about 230
// us.  Arrays from 32 KiB (uploads to 1 MiB, where the runtime's own pipeline
// is as fast) therefore go through pinned slots of the context's; arrays
// pinned by the caller, and any other memory the runtime knows (a device array
// in a host array's place), move directly.  Used with the context's lock held, on
// its stream.
class HostStage {
 public:
  static constexpr size_t kSlot = (size_t)1 << 20, kMin = (size_t)32 << 10;
  static constexpr int kSlots = 4;
  ~HostStage() {
    if (buf_) (void)hipHostFree(buf_);
  }
  Status init() {
    PSSA_HIP_TRY(hipHostMalloc(reinterpret_cast<void**>(&buf_), kSlot * kSlots, 0));
    return Status::Ok();
  }
  // A pageable source may be reused at return; the copy is ordered on the
  // stream.
  Status to_device(void* dst, const void* src, size_t n, hipStream_t st) {
    if (!n) return Status::Ok();
    if (n >= kMin && n < kSlot && !known(src)) {
      if (used_ + n > kSlot * kSlots) PSSA_RETURN_IF(wait(st));
      std::memcpy(buf_ + used_, src, n);
      src = buf_ + used_;
      used_ += (n + 255) & ~(size_t)255;
    }
    PSSA_HIP_TRY(hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, st));
    return Status::Ok();
  }
  // The data is in `dst` once the stream is waited for.
  Status to_host(void* dst, const void* src, size_t n, hipStream_t st) {
    if (!n) return Status::Ok();
    if (n < kMin || known(dst)) {
      PSSA_HIP_TRY(hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, st));
      return Status::Ok();  // no wait of its own: some microseconds of a small call
    }
    PSSA_RETURN_IF(wait(st));
    auto piece = [&](size_t off) { return n - off < kSlot ? n - off : kSlot; };
    auto issue = [&](size_t off) {
      return hipMemcpyAsync(buf_ + off / kSlot % 2 * kSlot, static_cast<const char*>(src) + off, piece(off),
                            hipMemcpyDeviceToHost, st);
    };
    PSSA_HIP_TRY(issue(0));
    for (size_t off = 0; off < n; off += kSlot) {
      PSSA_HIP_TRY(hipStreamSynchronize(st));  // this piece is in its slot
      if (off + kSlot < n) PSSA_HIP_TRY(issue(off + kSlot));
      std::memcpy(static_cast<char*>(dst) + off, buf_ + off / kSlot % 2 * kSlot, piece(off));
    }
    return Status::Ok();
  }
  // Waits for the stream; every transfer out of or into the slots has ended.
  Status wait(hipStream_t st) {
    PSSA_HIP_TRY(hipStreamSynchronize(st));
    used_ = 0;
    return Status::Ok();
  }

 private:
  // Not plain pageable memory: the host may not be able to read or write it.
  static bool known(const void* p) {
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    return at.type != hipMemoryTypeUnregistered;
  }
  char* buf_ = nullptr;
  size_t used_ = 0;  // bytes of the slots that uploads may still be reading
};

// Orders this wave's LDS writes before its subsequent LDS reads.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// fp32 -> bf16 bits, rounded to nearest even, on gfx950's v_cvt_pk_bf16_f32
// (one instruction per pair; the same bits as the integer rounding
// u + 0x7FFF + lsb for every finite value).
typedef __bf16 bf16x2_cvt_t __attribute__((ext_vector_type(2)));
typedef float f32x2_cvt_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t bf16x2_bits(float lo, float hi) {
  const f32x2_cvt_t v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_cvt_t));
}
__device__ __forceinline__ uint16_t bf16_bits_dev(float f) { return (uint16_t)bf16x2_bits(f, 0.0f); }

// RMSNorm of one row by one wave (src/pssa.rs:1080-1086).  Lane L holds
// x[4L + 256k .. +3] for k < RMS_V4 (zero past d; d % 4 == 0, rows 16-byte
// aligned); the squares are summed per lane in (k, component) order, then
// across the wave by the xor butterfly.  Every kernel that normalises rows
// (the standalone norm and the decode input product) goes through these two
// functions, so they agree bit for bit.
constexpr int RMS_V4 = 4;  // float4s per lane: rows of up to 1024 columns
__device__ __forceinline__ void rms_load_v4(const float* x, int d, int lane, float4 (&xv)[RMS_V4]) {
#pragma unroll
  for (int k = 0; k < RMS_V4; ++k) {
    const int i = 4 * lane + 256 * k;
    xv[k] = i < d ? *reinterpret_cast<const float4*>(x + i) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
}
// 1 / sqrt(mean square + 1e-5) of each of R rows a wave holds (rms_load_v4):
// per row the same chain, the rows' butterfly steps interleaved so their
// cross-lane exchanges are in flight together.
template <int R>
__device__ __forceinline__ void rms_inv_v4(const float4 (&xv)[R][RMS_V4], int d, float (&inv)[R]) {
  float ss[R];
#pragma unroll
  for (int q = 0; q < R; ++q) {
    ss[q] = 0.0f;
#pragma unroll
    for (int k = 0; k < RMS_V4; ++k) {
      ss[q] = fmaf(xv[q][k].x, xv[q][k].x, ss[q]);
      ss[q] = fmaf(xv[q][k].y, xv[q][k].y, ss[q]);
      ss[q] = fmaf(xv[q][k].z, xv[q][k].z, ss[q]);
      ss[q] = fmaf(xv[q][k].w, xv[q][k].w, ss[q]);
    }
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    float o[R];
#pragma unroll
    for (int q = 0; q < R; ++q) o[q] = __shfl_xor(ss[q], off, 64);
#pragma unroll
    for (int q = 0; q < R; ++q) ss[q] += o[q];
  }
#pragma unroll
  for (int q = 0; q < R; ++q) inv[q] = 1.0f / sqrtf(ss[q] / (float)d + 1e-5f);
}
// gamma * (x * inv) + beta, the multiply-add rounded once.
__device__ __forceinline__ float rms_apply(float x, float inv, float g, float b) { return fmaf(g, x * inv, b); }

// s_waitcnt immediate for vmcnt(v) alone (gfx9: vmcnt bits [3:0] and [15:14],
// expcnt and lgkmcnt left at their no-wait maxima).
constexpr int vmcnt_only(int v) { return (v & 0xF) | (((v >> 4) & 3) << 14) | (0x7 << 4) | (0xF << 8); }

}  // namespace pssa

// The opaque context handed out through the C ABI.
struct pssa_hip_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string name;
  int cu_count = 0;
  std::mutex mu;
  pssa::HostStage stage;
  pssa::DevPool pool;  // before every member whose buffers return to it
  // Kernel scratch reused across calls (grown on demand, freed with the
  // context); calls on one context are serialised by `mu` on one stream.
  void* scratch = nullptr;
  size_t scratch_bytes = 0;
  // Device address of this device's static scratch array (the
  // allocation-free retrieval), resolved when the context is created.
  void* noalloc_scratch = nullptr;
  // Device copies of GEMM weights keyed by (host address, element count,
  // storage dtype), as the reference's CUDA weight cache keys them by
  // (address, length).  A stale entry is uploaded again on its next use.
  struct CachedWeight {
    pssa::DevBuf buf;
    bool current = true;
  };
  std::map<std::tuple<uintptr_t, size_t, int>, CachedWeight> weights;
  // The SSM tape left on the device by pssa_hip_ssm_forward_resident for
  // the next pssa_hip_memory_forward_after_ssm (opaque here).
  std::shared_ptr<struct SsmTape> ssm_tape;
};
