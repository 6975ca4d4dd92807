// Copies between ordinary host memory and a device.
//
// A copy straight from or to pageable memory makes the runtime lock the pages
// for the transfer: 512 KiB took 210 us to the device and 250 us back, against
// 18 us through a page-locked block that is already there, and memory freed
// after such a copy stops the process's queues while the lock is dropped (a
// burst of requests to a server took 10 ms instead of 4).  Blocks are not
// allocated per call either: their first touch costs 0.19 us per KiB.  So each
// device context keeps 8 blocks of 2 MiB, touched once.  A host thread copies
// at about 30 GB/s and the link runs at about 55 GB/s, so copies of 4 MiB and
// more take up to 4 threads, two blocks each: one is on the link while the
// other is filled or emptied.  48 MB: 1.7 -> 1.0 ms to the device, 3.0 -> 1.0
// ms back.  Memory that is known to the runtime (page-locked or on a device) is
// copied directly.
//
// The blocks are one lock for every copy of a device, a server's submits among
// them, so nothing waits for a kernel while it holds them: copy_to_host waits for
// the stream first, and a copy to the device goes on a stream that no other call's
// kernels are queued on.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>

#include "capi_common.h"

namespace ppsk {
namespace capi {

namespace {

// Page-locked, managed or device memory: no staging needed.
bool known_memory(const void* p) {
  hipPointerAttribute_t at;
  if (hipPointerGetAttributes(&at, p) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return at.type != hipMemoryTypeUnregistered;
}

// Runs work(lane) on up to HostStage::LANES threads, the caller's included.  A
// thread that cannot be started leaves its pieces to the others.
template <typename F>
void on_lanes(int lanes, F work) {
  std::thread extra[HostStage::LANES];
  for (int l = 1; l < lanes; ++l) {
    try {
      extra[l] = std::thread(work, l);
    } catch (const std::system_error&) {
      break;
    }
  }
  work(0);
  for (auto& t : extra) {
    if (t.joinable()) t.join();
  }
}

int lanes_for(size_t bytes) {
  return bytes < 2 * HostStage::BLOCK ? 1 : (int)std::min<size_t>(HostStage::LANES, bytes / HostStage::BLOCK);
}

}  // namespace

void copy_host(void* dst, const void* src, size_t bytes) {
  std::atomic<size_t> next{0};
  on_lanes(lanes_for(bytes), [&](int) {
    for (size_t at; (at = next.fetch_add(HostStage::BLOCK)) < bytes;) {
      const size_t n = std::min(HostStage::BLOCK, bytes - at);
      if (src) std::memcpy((char*)dst + at, (const char*)src + at, n);
      else std::memset((char*)dst + at, 0, n);
    }
  });
}

hipError_t HostStage::init() {
  hipError_t e = hipSuccess;
  for (int x = 0; x < 2 * LANES && e == hipSuccess; ++x) {
    e = hipHostMalloc((void**)&block[x], BLOCK, hipHostMallocDefault);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&done[x], hipEventDisableTiming);
    if (e == hipSuccess) std::memset(block[x], 0, BLOCK);
  }
  return e;
}

hipError_t fill_device(DeviceCtx* c, void* dst, size_t bytes, hipStream_t stream, const Fill& fill) {
  if (bytes == 0) return hipSuccess;
  HostStage& h = c->host;
  std::lock_guard<std::mutex> lk(h.mu);
  std::atomic<size_t> next{0};
  std::atomic<int> err{hipSuccess};
  on_lanes(lanes_for(bytes), [&](int lane) {
    hipError_t e = hipSetDevice(c->device);
    for (int turn = 0; e == hipSuccess && err.load() == hipSuccess; turn ^= 1) {
      const size_t at = next.fetch_add(HostStage::BLOCK);
      if (at >= bytes) return;
      const size_t n = std::min(HostStage::BLOCK, bytes - at);
      const int x = 2 * lane + turn;
      e = hipEventSynchronize(h.done[x]);  // the block's last copy has left it
      if (e != hipSuccess) break;
      fill(h.block[x], at, n);
      e = hipMemcpyAsync((char*)dst + at, h.block[x], n, hipMemcpyHostToDevice, stream);
      if (e == hipSuccess) e = hipEventRecord(h.done[x], stream);
    }
    if (e != hipSuccess) err.store(e);
  });
  return (hipError_t)err.load();
}

hipError_t copy_to_device(DeviceCtx* c, void* dst, const void* src, size_t bytes,
                          hipStream_t stream) {
  if (bytes == 0) return hipSuccess;
  if (known_memory(src)) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream);
  return fill_device(c, dst, bytes, stream, [src](char* to, size_t at, size_t n) {
    std::memcpy(to, (const char*)src + at, n);
  });
}

hipError_t copy_to_host(DeviceCtx* c, void* dst, const void* src, size_t bytes,
                        hipStream_t stream) {
  if (bytes == 0) return hipSuccess;
  if (known_memory(dst)) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream);
    return e == hipSuccess ? hipStreamSynchronize(stream) : e;
  }
  if (stream != c->copy_stream) {  // (no kernels there, and waiting costs a first pass 40 us)
    if (const hipError_t e = hipStreamSynchronize(stream)) return e;
  }
  HostStage& h = c->host;
  std::lock_guard<std::mutex> lk(h.mu);
  std::atomic<size_t> next{0};
  std::atomic<int> err{hipSuccess};
  on_lanes(lanes_for(bytes), [&](int lane) {
    hipError_t e = hipSetDevice(c->device);
    size_t at[2] = {0, 0}, n[2] = {0, 0};  // the piece each block holds
    // the next piece into block x; the other lanes' copies on the stream may
    // lie between this lane's, never its own block's contents
    auto start = [&](int x) {
      n[x] = 0;
      const size_t a = next.fetch_add(HostStage::BLOCK);
      if (a >= bytes) return hipSuccess;
      at[x] = a;
      n[x] = std::min(HostStage::BLOCK, bytes - a);
      const int b = 2 * lane + x;
      hipError_t s = hipEventSynchronize(h.done[b]);
      if (s == hipSuccess) {
        s = hipMemcpyAsync(h.block[b], (const char*)src + a, n[x], hipMemcpyDeviceToHost, stream);
      }
      if (s == hipSuccess) s = hipEventRecord(h.done[b], stream);
      return s;
    };
    if (e == hipSuccess) e = start(0);
    for (int x = 0; e == hipSuccess && n[x] != 0; x ^= 1) {
      e = start(x ^ 1);
      if (e == hipSuccess) e = hipEventSynchronize(h.done[2 * lane + x]);
      if (e == hipSuccess) std::memcpy((char*)dst + at[x], h.block[2 * lane + x], n[x]);
    }
    if (e != hipSuccess) err.store(e);
  });
  // after an error nothing may still be on its way into the blocks
  if (err.load() != hipSuccess) (void)hipStreamSynchronize(stream);
  return (hipError_t)err.load();
}

}  // namespace capi
}  // namespace ppsk
