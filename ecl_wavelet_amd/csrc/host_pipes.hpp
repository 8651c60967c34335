// host_pipes.hpp -- what a host-issued batch works with (streams and pinned
// staging), and the pool that keeps it between calls.  The runtime comes in
// as Rt, so the pool's rules are tested without a device.
#pragma once

#include <algorithm>
#include <cstddef>
#include <memory>
#include <mutex>

namespace ecl {
namespace lib {

constexpr int kPipeSlots = 3;
constexpr int kPipeDevices = 64;
constexpr size_t kPipeMinBytes = size_t(1) << 20;  // smallest buffer of a slot
// Idle pipes kept per device: as many as may call at once without a pipe
// being made and unmade per call.  With four, 16 threads took twice as long
// as with a pipe per tree (rank batches of 10^5: 44 -> 78 us each).  A pipe
// has at most 36 MB pinned (3 slots of 2^19 queries of 16 bytes and results
// of 8), so 32 of them 1.2 GB; a pipe per tree had pinned 192 MB each.
constexpr size_t kIdlePipes = 32;

// Rt: Stream; Error, kOk and check(e, what), which throws for others;
// stream_create(Stream*), stream_destroy(Stream), pinned_alloc(void**,
// size_t), pinned_free(void*); DeviceScope(device).

template <class Rt>
class PipePool;

// kPipeSlots streams, each with pinned input and output buffers grown on
// demand
template <class Rt>
struct HostPipe {
  int device = 0;
  typename Rt::Stream stream[kPipeSlots] = {};
  void* pin_in[kPipeSlots] = {};
  void* pin_out[kPipeSlots] = {};
  size_t cap_in[kPipeSlots] = {}, cap_out[kPipeSlots] = {};

  HostPipe() = default;
  HostPipe(const HostPipe&) = delete;
  HostPipe& operator=(const HostPipe&) = delete;
  ~HostPipe() {
    for (int i = 0; i < kPipeSlots; ++i) {
      if (stream[i]) Rt::stream_destroy(stream[i]);
      if (pin_in[i]) Rt::pinned_free(pin_in[i]);
      if (pin_out[i]) Rt::pinned_free(pin_out[i]);
    }
  }
  void reserve(PipePool<Rt>& pool, int slots, size_t in_bytes, size_t out_bytes) {
    for (int i = 0; i < slots; ++i) {
      if (!stream[i]) Rt::check(Rt::stream_create(&stream[i]), "hipStreamCreate");
      grow(pool, pin_in[i], cap_in[i], in_bytes);
      grow(pool, pin_out[i], cap_out[i], out_bytes);
    }
  }

 private:
  static void grow(PipePool<Rt>& pool, void*& pin, size_t& cap, size_t bytes) {
    if (bytes <= cap) return;
    if (pin) Rt::pinned_free(pin);
    pin = nullptr;
    cap = 0;
    bytes = std::max(bytes, kPipeMinBytes);
    pin = pool.alloc_pinned(bytes);
    cap = bytes;
  }
};

// Idle pipes per device, shared by all trees and threads.
template <class Rt>
class PipePool {
 public:
  using Pipe = HostPipe<Rt>;

  // an idle pipe of the device, or a new one
  std::unique_ptr<Pipe> take(int device) {
    if (device >= 0 && device < kPipeDevices) {
      Idle& d = dev_[device];
      std::lock_guard<std::mutex> lk(d.mu);
      if (d.count) return std::move(d.pipe[--d.count]);
    }
    std::unique_ptr<Pipe> p(new Pipe());
    p->device = device;
    return p;
  }
  // keeps a pipe whose streams are idle, or frees it
  void give(std::unique_ptr<Pipe> p) noexcept {
    if (p->device < 0 || p->device >= kPipeDevices) return;
    Idle& d = dev_[p->device];
    std::lock_guard<std::mutex> lk(d.mu);
    if (d.count < kIdlePipes) d.pipe[d.count++] = std::move(p);
  }
  // frees the device's idle pipes
  void release(int device) noexcept {
    if (device < 0 || device >= kPipeDevices) return;
    std::unique_ptr<Pipe> gone[kIdlePipes];
    {
      Idle& d = dev_[device];
      std::lock_guard<std::mutex> lk(d.mu);
      for (size_t i = 0; i < d.count; ++i) gone[i] = std::move(d.pipe[i]);
      d.count = 0;
    }
    if (!gone[0]) return;
    typename Rt::DeviceScope ds(device);
    for (std::unique_ptr<Pipe>& p : gone) p.reset();
  }
  void release_all() noexcept {
    for (int d = 0; d < kPipeDevices; ++d) release(d);
  }
  // Pinned host memory.  When the runtime has none left, the idle pipes of
  // every device are given back and it is asked once more.
  void* alloc_pinned(size_t bytes) {
    void* p = nullptr;
    typename Rt::Error e = Rt::pinned_alloc(&p, bytes);
    if (e != Rt::kOk) {
      release_all();
      p = nullptr;
      e = Rt::pinned_alloc(&p, bytes);
    }
    Rt::check(e, "hipHostMalloc");
    return p;
  }

 private:
  struct Idle {
    std::mutex mu;
    std::unique_ptr<Pipe> pipe[kIdlePipes];
    size_t count = 0;
  };
  Idle dev_[kPipeDevices];
};

}  // namespace lib
}  // namespace ecl
